// Mixed block-scaled GEMM for gfx950 on v_mfma_scale_f32_16x16x128_f8f6f4.
//
//   D[m][n] = bf16( sum_seg sum_kb 2^(sfa-127) 2^(sfb-127) sum_{32} a*b )
//
// replacing the reference's three chained CUTLASS segment GEMMs
// (src/gemm.cu:44-46; src/fp4.cu:35, src/fp6.cu:35, src/fp8.cu:35): all three K
// segments (E2M1, E3M2, E4M3 activations against E2M1 weights) accumulate into
// one fp32 tile and D is rounded to bf16 once.
//
// The weights are fed as the MFMA's first operand and the activations as the
// second, so the 16x16 result tile is D^T: a lane ends up with four consecutive
// output features n of one token m, which are adjacent in row-major D.
//
// Operand geometry of the instruction (measured on gfx950): lane l supplies row
// i = l % 16 of its operand; with g = l / 16,
//   E2M1 / E3M2: the 32 consecutive K elements of block g of the 128-wide K
//                step -- one MX block, 16 or 24 contiguous bytes;
//   E4M3:        K elements [16g, 16g+16) in registers 0-3 and
//                [64+16g, 64+16g+16) in registers 4-7 (two 16-byte pieces);
// and, for every format, the E8M0 scale of block g of row i in the byte of the
// scale register that op_sel selects.
#include <math.h>

#include <type_traits>

#include "mg_common.h"
#include "quantize.h"
#include "tile_order.h"

namespace mg {

namespace {

template <int FMT>
struct Frag;
template <> struct Frag<kFmtE2M1> { static constexpr int kBytes = 16; };
template <> struct Frag<kFmtE3M2> { static constexpr int kBytes = 24; };
template <> struct Frag<kFmtE4M3> { static constexpr int kBytes = 32; };

// Up to four consecutive features n ... n + 3 of token m, rounded to bf16, with the epilogue's bias.
__device__ __forceinline__ void store4(uint16_t* __restrict__ d, const Epilogue& ep, int m, int n, v4f sum) {
  if (n >= ep.n_out) return;
  uint16_t h[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    h[v] = __builtin_bit_cast(uint16_t, (__bf16)sum[v]);
    if (ep.bias && n + v < ep.n_out) h[v] = add_bf16(h[v], ep.bias[n + v]);
  }
  uint16_t* dst = d + (size_t)m * ep.n_out + n;
  if (n + 3 < ep.n_out && (ep.n_out & 3) == 0 && (n & 3) == 0) {
    *reinterpret_cast<v2u*>(dst) = v2u{(unsigned)h[0] | ((unsigned)h[1] << 16), (unsigned)h[2] | ((unsigned)h[3] << 16)};
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (n + v < ep.n_out) dst[v] = h[v];
  }
}
// One feature.
__device__ __forceinline__ void store1(uint16_t* __restrict__ d, const Epilogue& ep, int m, int n, float sum) {
  if (n >= ep.n_out) return;
  uint16_t h = __builtin_bit_cast(uint16_t, (__bf16)sum);
  if (ep.bias) h = add_bf16(h, ep.bias[n]);
  d[(size_t)m * ep.n_out + n] = h;
}

// ---------------------------------------------------------------------------
// Skinny kernel: few tokens (decode, small batches), any 32-granular K, wherever the rules below do not find another kernel
// faster.  Weights are streamed once per 16 * G tokens (HBM- or L2-bound).
//
// A workgroup of 4 waves owns F groups of 16 output features and G groups of 16 tokens; the K steps (128 elements
// each, counted over the three segments) are dealt to the waves in contiguous quarters (as in the decode kernel below:
// the same sums in the same order, whichever of the two a shape goes to).  Each wave runs a pipeline of its own: a
// ring of NS slots in LDS, one step each (weight codes, token codes, the 16-byte pieces of the scale atoms that hold
// its rows), filled by global -> LDS copies NS - 1 steps ahead and refilled as soon as its fragments are in registers,
// whole steps two at a time: one wait for two steps' fragments.  Requests of whole steps are addresses that advance and offsets that
// stay; the steps around a segment's end, and the first ones, are addressed one by one.
// No barrier until the waves' partial 16x16 tiles are summed; nothing in flight occupies a register.
//
// What bounds it, from counters: a launch takes about 2.3 us + 0.07 ... 0.14 us per K step.  With few steps that is the
// latency of the first copies and of one step after the other (N = K = 4096: address unit busy 24 % of the kernel with 1
// token, 45 % with 128, the waves waiting 57 ... 62 % of their cycles); with many steps and tokens the address unit, at 26 ...
// 37 cycles per copy of 16 rows x 64 bytes (N = 4096, K = 14336: busy 47 % with 32 tokens, 66 % on row-major weights, 72 and 76 %
// with 128).  The matrix cores are busy 1 ... 8 %.  So the token fragments of a step are as many copies as their format has
// kilobytes, and all scales of a step are one copy.  The 16-byte pieces of a row are copied by neighbouring lanes and
// permuted inside the row (XOR with bits of the row number), so that the fragment reads spread over the LDS banks.
// Before (fragments and scale bytes loaded into registers, each round of steps waited for as a whole; tile-major weights
// of two layers in turn, K = 14336, N = 4096): M = 16 17.5 -> 11.0 us, 32 23 -> 12.2, 64 28 -> 13.1, 128 47 (whole-tile
// kernel) -> 16.8, 200 47 -> 30.8; K = 4096, N = 4096, M = 128 9.0 -> 7.9 (decode kernel with 32 tokens per workgroup,
// which this replaces).
// Layer call (quantizer and this kernel) from HBM, tile-major weights, us, with eight slots, one step at a time -> shorter rings 8.9, two
// steps at a time 8.75, all arguments fetched in one batch 8.55: M = 16, N = K = 4096 9.4 -> 8.55; M = 32, N = 4096, K = 14336 19.5 -> 18.3; M =
// 128, N = K = 4096 13.8 -> 13.1 (eight slots of the form with half the features before).  With what the kernel's constants say below, 400
// calls of 1 ... 255 tokens are 1.053 / 1.044 times as fast from the caches / from HBM as with eight slots, three and one of them slower by more than
// 2.5 % (two runs of one side differ by 2); slowest are row-major weights with four and eight feature groups, 0.996 ... 1.009 in the mean.
// ---------------------------------------------------------------------------
struct DecodeSeg {
  const uint8_t* a;
  const uint8_t* b;
  const uint8_t* sfa;
  const uint8_t* sfb;
  int nblk;    // 32-element blocks in the segment
  int steps;   // ceil(nblk / 4)
};

template <int FMT>
__device__ __forceinline__ v4f decode_mfma(v8i wb, v8i xa, v4f acc, int sw, int sx) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wb, xa, acc, kFmtE2M1, FMT, 0, sw, 0, sx);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

// waits until at most `steps` (wave-uniform, at most MOST) steps of PER copies each are in flight
template <int PER, int MOST>
__device__ __forceinline__ void wait_steps(int steps) {
  static_assert(MOST <= 4, "cases");
  switch (steps) {
#define MG_STEPS_CASE(N) case N: if constexpr (N <= MOST) { wait_vmcnt<N * PER>(); break; } [[fallthrough]];
    MG_STEPS_CASE(1) MG_STEPS_CASE(2) MG_STEPS_CASE(3) MG_STEPS_CASE(4)
#undef MG_STEPS_CASE
    default: wait_vmcnt<0>(); break;
  }
}

template <bool STREAM = false>
__device__ __forceinline__ void dma16_at(const uint8_t* base, unsigned voff, unsigned lds_off) {
  // base and lds_off are wave-uniform; say so to the compiler
  const uint64_t bv = reinterpret_cast<uint64_t>(base);
  // (the builtin returns int: without the casts the low half would be sign-extended over the high half)
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)bv);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(bv >> 32));
  base = reinterpret_cast<const uint8_t*>(((uint64_t)hi << 32) | lo);
  lds_off = __builtin_amdgcn_readfirstlane(lds_off);
  if constexpr (STREAM) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                                     : : "v"(voff), "s"(base), "s"(lds_off) : "memory", "m0");
  else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                    : : "v"(voff), "s"(base), "s"(lds_off) : "memory", "m0");
}
// the same with a 64-bit address per lane
__device__ __forceinline__ void dma16_lane(const uint8_t* p, unsigned lds_off) {
  lds_off = __builtin_amdgcn_readfirstlane(lds_off);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(p), "s"(lds_off) : "memory", "m0");
}

// copies of 1 KB per step for 16 G tokens of a format
template <int FMT, int G>
constexpr int kTokenCopies = (16 * G * 4 * Frag<FMT>::kBytes + 1023) / 1024;
// LDS bytes of a slot, and slots per wave.  Four slots, three where four do not fit: a wave that has more to request before its first step stands at
// its requests -- a CU takes no more than some 40 KB of them ahead of the data -- while the first steps' data is there.  Layer call, M = 16, N = K =
// 4096 from HBM with 3 / 4 / 5 / 6 / 8 / 12 slots 9.1 / 8.7 / 8.9 / 9.0 / 9.4 / 9.7 us, K = 14336 17.9 / 16.5 / 16.7 / 16.9 / 17.3 / 18.2.
template <int G, int F>
constexpr int kSkinnyPieces = (G == 1 ? 16 : 32) + 4 * F;   // scale pieces of a step: tokens, weights
template <int G, int F>
constexpr int kSkinnySlot = 1024 * (F + 2 * G) + 16 * kSkinnyPieces<G, F>;
template <int G, int F>
constexpr int kSkinnySlots = 159 * 1024 / (4 * kSkinnySlot<G, F>) < 4 ? 3 : 4;

// ONCE: launches of at most NS - 1 steps per wave, which are all requested up front.  One step at a time and nothing requested in the loop: with
// less code around them so few steps end sooner (172 layer calls of 3 steps per wave, K < 2000, against the pipeline's form from the caches /
// from HBM 1.8 % / 1.6 % faster, in pairs 0.8 % each; both loops in one kernel made the longer launches 5 % slower).
template <int G, int F, bool WT, bool ONCE>
__global__ void __launch_bounds__(256)
mixed_gemm_skinny_kernel(DecodeSeg s4, DecodeSeg s6, DecodeSeg s8, int M, int N, int steps_per_wave, TileOrder order,
                         Epilogue ep, uint16_t* __restrict__ d) {
  constexpr int NS = kSkinnySlots<G, F>, kSlot = kSkinnySlot<G, F>;
  constexpr int PA = G == 1 ? 16 : 32, PB = 4 * F;   // scale pieces per step: tokens, weights
  // The widest layers' weight codes, whole lines that nobody reads again, as streaming loads: they leave the last-level cache to
  // what follows.  N = 28672, K = 4096, M = 16 from HBM 15.3 -> 14.2 us, 20480 13.4 -> 12.7 (from that cache 12.3 -> 13.3); a decoder
  // layer's four projections of 16 tokens, whose others (58 MB) then stay in it, 62.5 -> 56.3.
  constexpr bool kStream = WT && F == 8;
  constexpr int kScales = 1024 * (F + 2 * G);   // where a slot's scales begin
  // Whole steps two at a time where the ring has four slots.  Out of three, with one step in flight, pairs are slower (N = 20480, K = 5120, M =
  // 16 18.5 against 18.0 us), and so they are with two token and four feature groups on row-major weights, where the copies of half
  // lines are what a step waits for (24 calls, from HBM / from the caches 1.5 % and 1.4 % faster one at a time; M = 20, N = 11264, K = 2496 9.1 -> 8.8).
  constexpr bool kPairs = !ONCE && NS > 3 && (WT || G != 2 || F != 4);
  // Requests of whole steps by advancing addresses, which single steps out of three slots use on row-major weights alone: on tile-major ones
  // both ways of addressing are more scalars than there are (8 and 9 were spilled; 24 calls of (1, 8) 1.0 % and 1.8 % faster without).
  constexpr bool kAdvance = !ONCE && (NS > 3 ? kPairs : !WT);
  // A wave's last NS - 1 steps are waited for at once, or (four and eight feature groups, whose steps are 4 and 8 KB of weights) each by
  // itself: 200 layer calls of K < 2000, the steps each by itself over at once from HBM / from the caches, (1, 1) 1.4 % and 0.9 % slower,
  // (1, 2) level / 0.3 % slower, (1, 4) 1.2 % faster / 0.9 % slower, (2, 4) 1.5 % faster / 0.9 % slower.
  constexpr bool kLastAtOnce = F < 4;
  static_assert(NS >= 3 && PA + PB <= 64, "a pipeline; one copy for all scales of a step");
  extern __shared__ __align__(16) uint8_t lds[];
  // all arguments in one batch of loads (see pin_args)
  asm volatile("" : : "s"(s4.a), "s"(s4.sfb), "s"(s4.nblk), "s"(s4.steps), "s"(s6.a), "s"(s6.sfb), "s"(s6.nblk), "s"(s6.steps), "s"(s8.a),
               "s"(s8.sfb), "s"(s8.nblk), "s"(s8.steps), "s"(M), "s"(N), "s"(steps_per_wave), "s"(order.xlog), "s"(order.magic),
               "s"(order.tiles), "s"(ep.bias), "s"(ep.n_out), "s"(d));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  uint8_t* const ring = lds + wave * (NS * kSlot);
  const unsigned ring0 = (unsigned)(size_t)(__attribute__((address_space(3))) uint8_t*)lds + (unsigned)wave * (NS * kSlot);
  const int t6 = s4.steps, t8 = s4.steps + s6.steps, total = t8 + s8.steps;
  const int t_begin = wave * steps_per_wave, t_end = min(total, t_begin + steps_per_wave);

  // ---- the workgroup's rows: the mapping of the decode kernel below (feature group f, lane row i -> its scale piece
  // and its dword in the piece), and the weight row this lane copies, row lane / 4 of the group
  // (an XCD has runs of workgroups: those of the same features, for other tokens, find the weights in its L2 -- M = 19, N = 7424, K =
  // 18944, whose two token groups were on different XCDs, 31.9 -> 28.0 us --, and those of a 256-feature tile of tile-major weights
  // put their sectors of the result together there, see the decode kernel)
  const int launched = (int)blockIdx.x + order.grid_x * (int)blockIdx.y;
  if (launched >= order.tiles) return;
  int wg, token_group;
  tile_at(order, launched, wg, token_group);
  constexpr int per_group = 32 / PB;
  const int tile = (wg * F) >> 4, j0 = (wg * F) & 15;                    // tile-major
  const int group = wg / per_group, c0 = (wg % per_group) * PB;          // row-major
  auto feature = [&](int f, int e) {   // feature e of group f
    if constexpr (WT) return tile * 256 + j0 + f + 32 * (e & 7) + 16 * (e >> 3);
    else return group * 128 + c0 + (16 * f + e) % PB + 32 * ((16 * f + e) / PB);
  };
  int sw_off[F];   // this lane's weight scale byte in a step's pieces
  int wrow[F];     // the weight row it copies
#pragma unroll
  for (int f = 0; f < F; ++f) {
    if constexpr (WT) sw_off[f] = (PA + (((i & 7) >> 2) * 2 + (i >> 3)) * F + f) * 16 + (i & 3) * 4 + g;
    else sw_off[f] = (PA + (16 * f + i) % PB) * 16 + ((16 * f + i) / PB) * 4 + g;
    wrow[f] = min(feature(f, lane >> 2), N - 1);   // rows past N: read again, never stored
  }
  const int m_base = token_group * 16 * G, last_row = min(M - m_base, 16 * G) - 1;
  // the scale piece this lane copies, as an address in each segment's first step
  const uint8_t *sc4, *sc6, *sc8;
  {
    const int pl = min(lane, PA + PB - 1) - PA;
    unsigned piece;
    int mul;
    if (pl < 0) {
      piece = (unsigned)((m_base & 31) + pl + PA);
      mul = m_base >> 7;
    } else if constexpr (WT) {
      piece = (unsigned)(j0 + pl % F + 16 * ((pl / F) & 1));
      mul = tile * 2 + pl / (2 * F);
    } else {
      piece = (unsigned)(c0 + pl);
      mul = group;
    }
    sc4 = (pl < 0 ? s4.sfa : s4.sfb) + (size_t)mul * s4.steps * 512 + piece * 16;
    sc6 = (pl < 0 ? s6.sfa : s6.sfb) + (size_t)mul * s6.steps * 512 + piece * 16;
    sc8 = (pl < 0 ? s8.sfa : s8.sfb) + (size_t)mul * s8.steps * 512 + piece * 16;
  }

  // ---- requests step q of a segment into a slot
  const int wpos = (lane & 3) ^ ((lane >> 4) & 3);   // the 16-byte piece of its row that this lane copies
  auto request_seg = [&](auto fmt_c, const DecodeSeg& s, const uint8_t* sc, int q, unsigned slot) __attribute__((always_inline)) {
    constexpr int FMT = decltype(fmt_c)::value;
    const int left = min(s.nblk - 4 * q, 4);
    if (lane < kSkinnyPieces<G, F>) dma16_lane(sc + (size_t)q * 512, slot + kScales);
    const unsigned wp = (unsigned)min(wpos, left - 1) * 16u;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const unsigned at = slot + 1024u * f;
      if constexpr (WT) {
        // 16 KB per (256-feature tile, whole step), the group's block in it; the blocks past the last whole step as
        // rows of nblk % 4 blocks behind the tiled part
        const int whole = s.nblk >> 2;
        if (q < whole) dma16_at<kStream>(s.b + (((size_t)tile * whole + q) * 16 + j0 + f) * 1024, (unsigned)(lane >> 2) * 64u + wp, at);
        else dma16_at(s.b + (size_t)(N >> 8) * whole * 16384, (unsigned)wrow[f] * (unsigned)(s.nblk & 3) * 16u + wp, at);
      } else {
        dma16_at(s.b + (size_t)q * 64, (unsigned)wrow[f] * (unsigned)s.nblk * 16u + wp, at);
      }
    }
    const unsigned pitch = (unsigned)s.nblk * Frag<FMT>::kBytes;
    const uint8_t* a = s.a + (size_t)m_base * pitch + (size_t)q * (4 * Frag<FMT>::kBytes);
    constexpr int kPieces = Frag<FMT>::kBytes / 4;   // 16-byte pieces of a row's step
#pragma unroll
    for (int c = 0; c < kTokenCopies<FMT, G>; ++c) {
      const int chunk = min(c * 64 + lane, 16 * G * kPieces - 1), row = chunk / kPieces, p = chunk % kPieces;
      unsigned off;
      if constexpr (FMT == kFmtE2M1) off = (unsigned)min(p ^ ((row >> 2) & 3), left - 1) * 16u;
      else if constexpr (FMT == kFmtE3M2) off = (unsigned)min(p * 16, left * 24 - 16);
      else off = (unsigned)min(p ^ (row & 7), 2 * left - 1) * 16u;
      dma16_at(a, (unsigned)min(row, last_row) * pitch + off, slot + 1024u * (F + c));
    }
  };
  auto request = [&](int t, unsigned slot) __attribute__((always_inline)) {
    if (t >= t_end) return;
    if (t < t6) request_seg(std::integral_constant<int, kFmtE2M1>{}, s4, sc4, t, slot);
    else if (t < t8) request_seg(std::integral_constant<int, kFmtE3M2>{}, s6, sc6, t - t6, slot);
    else request_seg(std::integral_constant<int, kFmtE4M3>{}, s8, sc8, t - t8, slot);
  };

  v4f acc[F][G];
#pragma unroll
  for (int f = 0; f < F; ++f)
#pragma unroll
    for (int gi = 0; gi < G; ++gi) acc[f][gi] = v4f{0.f, 0.f, 0.f, 0.f};
  int sx_off[G];   // this lane's token scale byte in a step's pieces
#pragma unroll
  for (int gi = 0; gi < G; ++gi) {
    const int m = m_base + 16 * gi + i;
    sx_off[gi] = ((m - m_base) & (PA - 1)) * 16 + ((m >> 5) & 3) * 4 + g;
  }

  int t = t_begin, slot = 0;
#pragma unroll
  for (int k = 0; k < NS - 1; ++k) request(t_begin + k, ring0 + k * kSlot);
  if constexpr (ONCE && kLastAtOnce) wait_vmcnt<0>();
  // the fragments of a step in a slot
  struct Fragments { v4i w[F]; v8i x[G]; int s_w[F], s_x[G]; };
  const int frag4 = i * 64 + (g ^ ((i >> 2) & 3)) * 16;   // of 64-byte rows
  auto read = [&](auto fmt_c, Fragments& r, const uint8_t* sl, int left) __attribute__((always_inline)) {
    constexpr int FMT = decltype(fmt_c)::value;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      r.s_w[f] = sl[kScales + sw_off[f]];
      r.w[f] = *reinterpret_cast<const v4i*>(sl + 1024 * f + frag4);
    }
#pragma unroll
    for (int gi = 0; gi < G; ++gi) {
      r.s_x[gi] = sl[kScales + sx_off[gi]];
      const uint8_t* row = sl + 1024 * F + (16 * gi) * (4 * Frag<FMT>::kBytes);
      if constexpr (FMT == kFmtE2M1) {
        const v4i a = *reinterpret_cast<const v4i*>(row + frag4);
        r.x[gi] = v8i{a[0], a[1], a[2], a[3], 0, 0, 0, 0};
      } else if constexpr (FMT == kFmtE3M2) {
        const v2i* p = reinterpret_cast<const v2i*>(row + i * 96 + g * 24);
        // a partial step of 24 or 72 bytes: its last 16 bytes were copied, of which these are the second half
        const v2i a = p[0], b = p[1], e = p[(left & 1) && g == left - 1 ? 3 : 2];
        r.x[gi] = v8i{a[0], a[1], b[0], b[1], e[0], e[1], 0, 0};
      } else {   // K [16g, 16g+16) and [64+16g, 64+16g+16)
        const v4i a = *reinterpret_cast<const v4i*>(row + i * 128 + (g ^ (i & 7)) * 16);
        const v4i b = *reinterpret_cast<const v4i*>(row + i * 128 + ((4 + g) ^ (i & 7)) * 16);
        r.x[gi] = v8i{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      }
    }
  };
  auto multiply = [&](auto fmt_c, const Fragments& r) __attribute__((always_inline)) {
    constexpr int FMT = decltype(fmt_c)::value;
#pragma unroll
    for (int gi = 0; gi < G; ++gi)
#pragma unroll
      for (int f = 0; f < F; ++f)
        acc[f][gi] = decode_mfma<FMT>(v8i{r.w[f][0], r.w[f][1], r.w[f][2], r.w[f][3], 0, 0, 0, 0}, r.x[gi], acc[f][gi], r.s_w[f], r.s_x[gi]);
  };
  // the wave's steps of one segment
  auto run = [&](auto fmt_c, const DecodeSeg& s, const uint8_t* sc, int t_first, int t_next) __attribute__((always_inline)) {
    constexpr int FMT = decltype(fmt_c)::value, TC = kTokenCopies<FMT, G>, PER = 1 + F + TC;
    const int last = min(t_next, t_end);
    if (t >= last) return;
    const int whole = s.nblk >> 2, whole_end = min(last, t_first + whole);   // steps before whole_end are whole ones
    // Requests of whole steps of this segment, which most are: addresses that advance, and offsets that stay.
    const int q_next = t + NS - 1 - t_first;
    const uint8_t* sc_next = sc + (ptrdiff_t)q_next * 512;
    const uint8_t* w_next = WT ? s.b + (((ptrdiff_t)tile * whole + q_next) * 16 + j0) * 1024 : s.b + (ptrdiff_t)q_next * 64;
    const unsigned pitch = (unsigned)s.nblk * Frag<FMT>::kBytes;
    const uint8_t* a_next = s.a + (size_t)m_base * pitch + (ptrdiff_t)q_next * (4 * Frag<FMT>::kBytes);
    unsigned w_off[F], a_off[TC];
    if (kAdvance && t + NS - 1 < whole_end) {
#pragma unroll
      for (int f = 0; f < F; ++f) w_off[f] = WT ? (unsigned)(lane >> 2) * 64u + wpos * 16u : (unsigned)wrow[f] * (unsigned)s.nblk * 16u + wpos * 16u;
#pragma unroll
      for (int c = 0; c < TC; ++c) {
        constexpr int kPieces = Frag<FMT>::kBytes / 4;
        const int chunk = min(c * 64 + lane, 16 * G * kPieces - 1), row = chunk / kPieces, p = chunk % kPieces;
        a_off[c] = (unsigned)min(row, last_row) * pitch + (FMT == kFmtE2M1 ? p ^ ((row >> 2) & 3) : FMT == kFmtE3M2 ? p : p ^ (row & 7)) * 16u;
      }
    }
    auto next = [&](int ahead, unsigned to) __attribute__((always_inline)) {
      if constexpr (ONCE) return;
      if (kAdvance && ahead < whole_end) {
        if (lane < kSkinnyPieces<G, F>) dma16_lane(sc_next, to + kScales);
#pragma unroll
        for (int f = 0; f < F; ++f) dma16_at<kStream>(WT ? w_next + f * 1024 : w_next, w_off[f], to + 1024u * f);
#pragma unroll
        for (int c = 0; c < TC; ++c) dma16_at(a_next, a_off[c], to + 1024u * (F + c));
        sc_next += 512;
        w_next += WT ? 16384 : 64;
        a_next += 4 * Frag<FMT>::kBytes;
      } else {
        request(ahead, to);
      }
    };
    // Waits for steps t ... t + STEPS - 1, those up to t + NS - 1 requested: a wait counts the steps behind, each with at least as
    // many copies as this segment's (a token takes more bytes in every later segment's format).
    auto wait_for = [&](auto steps_c) __attribute__((always_inline)) {
      constexpr int kSteps = decltype(steps_c)::value;
      if constexpr (ONCE && kLastAtOnce) return;
      if (!ONCE && t + NS - 1 < t_end) wait_vmcnt<(NS - kSteps) * PER>();
      else if constexpr (kLastAtOnce) wait_vmcnt<0>();
      else wait_steps<PER, NS - 1 - kSteps>(t_end - kSteps - t);
    };
    while (t < last) {
      const uint8_t* sl = ring + slot * kSlot;
      const unsigned freed = ring0 + (unsigned)(slot == 0 ? NS - 1 : slot - 1) * kSlot;   // read a step ago
      if (kPairs && t + 1 < whole_end) {
        const int after = slot == NS - 1 ? 0 : slot + 1;
        const unsigned this_slot = ring0 + (unsigned)slot * kSlot;
        next(t + NS - 1, freed);
        wait_for(std::integral_constant<int, 2>{});
        Fragments r0, r1;
        read(fmt_c, r0, sl, 4);
        read(fmt_c, r1, ring + after * kSlot, 4);
        // the fragments are in registers before a later request may fill these slots again
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        next(t + NS, this_slot);
        multiply(fmt_c, r0);
        multiply(fmt_c, r1);
        slot = after == NS - 1 ? 0 : after + 1;
        t += 2;
      } else {
        next(t + NS - 1, freed);
        wait_for(std::integral_constant<int, 1>{});
        slot = slot == NS - 1 ? 0 : slot + 1;
        const int left = s.nblk - 4 * (t - t_first);
        Fragments r;
        read(fmt_c, r, sl, left);
        if (left < 4) {   // wave-uniform: the segment's last, partial step; what lies past its end is zero
          const bool ok = g < left, lo_ok = FMT == kFmtE4M3 ? (g >> 1) < left : ok, hi_ok = FMT == kFmtE4M3 ? 2 + (g >> 1) < left : ok;
#pragma unroll
          for (int f = 0; f < F; ++f) {
            r.s_w[f] = ok ? r.s_w[f] : 127;
#pragma unroll
            for (int e = 0; e < 4; ++e) r.w[f][e] = ok ? r.w[f][e] : 0;
          }
#pragma unroll
          for (int gi = 0; gi < G; ++gi) {
            r.s_x[gi] = ok ? r.s_x[gi] : 127;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              r.x[gi][e] = lo_ok ? r.x[gi][e] : 0;
              r.x[gi][4 + e] = hi_ok ? r.x[gi][4 + e] : 0;
            }
          }
        }
        if constexpr (!ONCE) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        multiply(fmt_c, r);
        ++t;
      }
    }
  };
  run(std::integral_constant<int, kFmtE2M1>{}, s4, sc4, 0, t6);
  run(std::integral_constant<int, kFmtE3M2>{}, s6, sc6, t6, t8);
  run(std::integral_constant<int, kFmtE4M3>{}, s8, sc8, t8, total);

  // ---- sum the four waves' partial tiles (D^T: lane holds token lane % 16, features 4 * (lane / 16) + v of a group)
  __syncthreads();   // every wave is done with its ring, which nothing fills any more
  float* partial = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int f = 0; f < F; ++f)
#pragma unroll
    for (int gi = 0; gi < G; ++gi)
      *reinterpret_cast<v4f*>(partial + ((wave * (F * G) + f * G + gi) * 64 + lane) * 4) = acc[f][gi];
  __syncthreads();
#pragma unroll
  for (int fg = 0; fg < F * G; ++fg) {
    if ((fg & 3) != wave) continue;
    const int f = fg / G, gi = fg % G;
    v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) sum += *reinterpret_cast<const v4f*>(partial + ((w * (F * G) + fg) * 64 + lane) * 4);
    const int m = m_base + 16 * gi + i;
    if (m < M) {
      if constexpr (WT) {
#pragma unroll
        for (int v = 0; v < 4; ++v) store1(d, ep, m, feature(f, 4 * g + v), sum[v]);
      } else {
        store4(d, ep, m, feature(f, 4 * g), sum);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Decode kernel: up to 16 tokens, whole 128-wide K steps.
//
// The skinny kernel above copies every step's token codes and scales for itself, for 16 tokens whether they exist or
// not: as many copies as the weights need.  Here everything that is not a weight code goes global -> LDS once per
// workgroup in 1 KB copies (global_load_lds_dwordx4): the token codes of all three segments (M x 2464 bytes for
// K = 4096) and, per K step, the 16-byte pieces of the scale
// atoms that hold the workgroup's rows; the K loop reads them from LDS.  The weight codes go to registers,
// eight K steps per wave at a time, in two rounds of four.  All
// requests are inline assembly, so that the waits can count them (requests complete in order).
//
// Which features a workgroup owns follows the scale atoms: a 16-byte piece of an atom holds rows c, c + 32,
// c + 64, c + 96 of a group of 128 (c = row % 32).  Row-major weights: the workgroup of 16 F features takes
// pieces c0 ... c0 + 4F - 1 of one group, i.e. rows c0 + (i % (4F)) + 32 (i / (4F)) for i = 0 ... 16F - 1 (its
// results are still runs of four consecutive features).  Tile-major weights: a workgroup takes F of the 1 KB
// copy blocks of a 256-feature tile (rows j + 32 t + 16 u, t = 0..7, u = 0, 1), whose scales are pieces j and
// j + 16 of both groups of the tile.  Either way the scales of a step are 64 F contiguous-by-piece bytes.
//
// Workgroup = 4 waves; the K steps (over the three segments) are dealt to the waves in contiguous quarters;
// partial tiles are summed through LDS.
// ---------------------------------------------------------------------------
struct DecodeLds {
  int x0, x1, x2;        // byte offsets of the token codes per segment
  int sfa0, sfa1, sfa2;  // of the token scale pieces: per step pa pieces of 16 bytes (piece p: tokens p, p + 32, p + 64, p + 96 of a group of 128)
  int sfb0, sfb1, sfb2;  // of the weight scale pieces: per step 4 F pieces
  int partial;           // of the partial sums
  int total;
  int pa;                // 8 (up to 8 tokens) or 16
};

// value of segment seg (0, 1, 2) by masking: a select between struct fields invites the compiler to index a private
// copy of the struct, which lands in scratch memory
__device__ __forceinline__ int sel3(int seg, int v0, int v1, int v2) {
  return (v0 & (seg == 0 ? -1 : 0)) | (v1 & (seg == 1 ? -1 : 0)) | (v2 & (seg == 2 ? -1 : 0));
}
__device__ __forceinline__ const uint8_t* sel3p(int seg, const uint8_t* p0, const uint8_t* p1, const uint8_t* p2) {
  const uint64_t m0 = seg == 0 ? ~0ull : 0ull, m1 = seg == 1 ? ~0ull : 0ull, m2 = seg == 2 ? ~0ull : 0ull;
  return reinterpret_cast<const uint8_t*>((reinterpret_cast<uint64_t>(p0) & m0) | (reinterpret_cast<uint64_t>(p1) & m1) |
                                          (reinterpret_cast<uint64_t>(p2) & m2));
}

// Copies `bytes` (a multiple of 16) from src to LDS offset dst in units of 1 KB, unit u by wave u % W; lanes past
// the end copy the last 16 bytes again (into the padding that rounds every region up to whole units).
template <int W = 4>
__device__ __forceinline__ void copy_region(const uint8_t* src, int bytes, unsigned dst, int wave, int lane) {
  const int units = (bytes + 1023) >> 10, chunks = bytes >> 4;
  for (int u = wave; u < units; u += W)
    dma16_at(src, (unsigned)min(u * 64 + lane, chunks - 1) * 16u, dst + (unsigned)u * 1024u);
}

// Copies P (4, 8 or 16, a power of two) 16-byte pieces per K step of a segment's scale atoms (512 bytes per step)
// to LDS as [step][piece]; piece_off is this lane's piece (lane % P) as a byte offset inside the atom (and, for
// pieces of another group of 128 rows, that group's distance).  Units of 1 KB = 64 / P steps, unit u by wave u % W;
// steps past the last one copy it again (into the region's padding).
// P = 1 << plog pieces per step (a power of two: no divisions by a run-time value here)
template <int W = 4>
__device__ __forceinline__ void copy_pieces(const uint8_t* src, int steps, int plog, unsigned piece_off, unsigned dst,
                                            int wave, int lane) {
  const int per_unit = 64 >> plog, units = (steps + per_unit - 1) >> (6 - plog);
  for (int u = wave; u < units; u += W) {
    const int q = min(u * per_unit + (lane >> plog), steps - 1);
    dma16_at(src, (unsigned)q * 512u + piece_off, dst + (unsigned)u * 1024u);
  }
}

// All arguments into scalar registers in one batch of loads: fetched where they are first used they cost a round trip
// to the argument buffer each time, before the first weight is requested.  The first statement wants one of every load's
// values at once (an input operand each; an in-out operand counts as two, and thirty is the limit), the others keep the
// compiler from fetching any of them again.
__device__ __forceinline__ void pin_args(DecodeSeg& s4, DecodeSeg& s6, DecodeSeg& s8, DecodeLds& l, int& M, int& N,
                                         int& steps_per_wave, Epilogue& ep, uint16_t* __restrict__& d) {
  asm volatile("" : : "s"(s4.a), "s"(s4.sfb), "s"(s4.nblk), "s"(s4.steps), "s"(s6.a), "s"(s6.sfb), "s"(s6.nblk), "s"(s6.steps),
               "s"(s8.a), "s"(s8.sfb), "s"(s8.nblk), "s"(s8.steps), "s"(M), "s"(N), "s"(steps_per_wave), "s"(l.x0), "s"(l.sfa0),
               "s"(l.sfb0), "s"(l.partial), "s"(l.pa), "s"(ep.bias), "s"(ep.n_out), "s"(d));
  asm volatile("" : "+s"(s4.a), "+s"(s4.b), "+s"(s4.sfa), "+s"(s4.sfb), "+s"(s4.nblk), "+s"(s4.steps));
  asm volatile("" : "+s"(s6.a), "+s"(s6.b), "+s"(s6.sfa), "+s"(s6.sfb), "+s"(s6.nblk), "+s"(s6.steps));
  asm volatile("" : "+s"(s8.a), "+s"(s8.b), "+s"(s8.sfa), "+s"(s8.sfb), "+s"(s8.nblk), "+s"(s8.steps));
  asm volatile("" : "+s"(l.x0), "+s"(l.x1), "+s"(l.x2), "+s"(l.sfa0), "+s"(l.sfa1), "+s"(l.sfa2), "+s"(l.sfb0), "+s"(l.sfb1),
               "+s"(l.sfb2), "+s"(l.partial), "+s"(l.total), "+s"(l.pa));
  asm volatile("" : "+s"(M), "+s"(N), "+s"(steps_per_wave), "+s"(d), "+s"(ep.bias), "+s"(ep.n_out));
}

// 16 bytes global -> registers as an instruction the compiler does not count; use after s_waitcnt + tie()
__device__ __forceinline__ void load16_uncounted(v4i& dst, const uint8_t* p) {
  asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(dst) : "v"(p) : "memory");
}
// the same from a wave-uniform base (scalar registers), a 32-bit per-lane offset and an immediate: one instruction
// per load and no 64-bit per-lane address arithmetic in front of it.  STREAM: as a streaming (nt) load -- the weight
// codes are read once; measured on tile-major weights 8.85 -> 8.70 us (N = 14336, K = 4096), on row-major ones, whose
// 64-byte row pieces share cache lines between K steps, 9.6 -> 9.9 us.
template <int OFF, bool STREAM = false>
__device__ __forceinline__ void load16_uncounted(v4i& dst, const uint8_t* sbase, unsigned voff) {
  static_assert(OFF >= 0 && OFF < 4096, "immediate offset of a global load");
  const uint64_t v = reinterpret_cast<uint64_t>(sbase);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  const uint64_t u = ((uint64_t)hi << 32) | lo;
  if constexpr (STREAM) asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3 nt" : "=v"(dst) : "v"(voff), "s"(u), "n"(OFF) : "memory");
  else asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(dst) : "v"(voff), "s"(u), "n"(OFF) : "memory");
}
__device__ __forceinline__ void tie(v4i& r) { asm volatile("" : "+v"(r)); }

// f of the integral constants N ... END - 1
template <int N, int END, class Fn>
__device__ __forceinline__ void for_each_step(Fn f) {
  if constexpr (N < END) {
    f(std::integral_constant<int, N>{});
    for_each_step<N + 1, END>(f);
  }
}

template <int F, bool WT>
__global__ void __launch_bounds__(256)
mixed_gemm_decode_kernel(DecodeSeg s4, DecodeSeg s6, DecodeSeg s8, int M, int N, int steps_per_wave, DecodeLds L,
                         Epilogue ep, uint16_t* __restrict__ d) {
  constexpr int S = 4;        // K steps per round
  constexpr int PB = 4 * F;   // weight scale pieces per step
  constexpr int PBLOG = F == 1 ? 2 : (F == 2 ? 3 : 4);
  static_assert(F == 1 || F == 2 || F == 4, "pieces per step as a power of two");
  extern __shared__ __align__(16) uint8_t lds[];
  pin_args(s4, s6, s8, L, M, N, steps_per_wave, ep, d);
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  // the segments' fields as scalars (selected by masks below, never by indexing)
  const uint8_t *b4 = s4.b, *b6 = s6.b, *b8 = s8.b;
  const int nblk4 = s4.nblk, nblk6 = s6.nblk, nblk8 = s8.nblk;
  const int total = s4.steps + s6.steps + s8.steps;
  const int t_begin = wave * steps_per_wave, t_end = min(total, t_begin + steps_per_wave);
  const int rounds = (t_end - t_begin + S - 1) / S;   // may be <= 0 for the last wave

  // ---- the workgroup's rows.  Feature group f, lane row i -> row n[f], its scale piece and its slot in the piece.
  int n[F], piece[F], slot[F];
  unsigned sfb_piece_off;   // this lane's piece (lane % PB) of the copies, as a byte offset from the segment's buffer
  int sfb_katoms_mul;       // ... plus this many times katoms * 512 (the piece's group of 128 rows)
  // Tile-major weights: which F blocks of which 256-feature tile.  The 16 / F workgroups of a tile each write 2 F of
  // every 16 consecutive output features, i.e. a part of every 32-byte sector of the tile's columns; workgroups go to
  // the 8 XCDs (one L2 each) round-robin by index, so the workgroups of a tile are given indices of one XCD, whose L2
  // then puts the sectors together instead of four L2s writing a part each (c2: 0.9 -> 0.23 MB written).
  int wg = blockIdx.x;
  if constexpr (WT) {
    constexpr int kPer = 16 / F;   // workgroups per tile
    if ((int)gridDim.x % (8 * kPer) == 0) {
      const int xcd = wg & 7, slot = wg >> 3;
      wg = ((slot / kPer) * 8 + xcd) * kPer + slot % kPer;
    }
  }
  if constexpr (WT) {
    // blocks j0 + f of tile `tile`; pieces ordered [group of 128][u][f]
    const int tile = (wg * F) >> 4, j0 = (wg * F) & 15;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const int t = i & 7, u = i >> 3;
      n[f] = tile * 256 + j0 + f + 32 * t + 16 * u;
      piece[f] = (t >> 2) * 2 * F + u * F + f;
      slot[f] = t & 3;
    }
    const int pl = lane % PB, pf = pl % F, pu = (pl / F) & 1, pg = pl / (2 * F);
    sfb_piece_off = (unsigned)(j0 + pf + 16 * pu) * 16u;
    sfb_katoms_mul = tile * 2 + pg;
  } else {
    // pieces c0 ... c0 + PB - 1 of group blockIdx.x / (32 / PB)
    const int per_group = 32 / PB, group = blockIdx.x / per_group, c0 = (blockIdx.x % per_group) * PB;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const int e = 16 * f + i;   // 0 ... 16 F - 1
      n[f] = group * 128 + c0 + e % PB + 32 * (e / PB);
      piece[f] = e % PB;
      slot[f] = e / PB;
    }
    sfb_piece_off = (unsigned)(c0 + lane % PB) * 16u;
    sfb_katoms_mul = group;
  }

  // ---- weight codes: per lane 16 bytes per step and feature group (row n[f], block g of the step)
  int nc[F];
#pragma unroll
  for (int f = 0; f < F; ++f) nc[f] = min(n[f], N - 1);   // clamped rows: every load is in bounds
  v4i wq[2][S][F];
  // Per-lane byte offsets of the loads.  Tile-major: 16 KB per (256-feature tile, step), the workgroup's F blocks of
  // 1 KB consecutive in it, lane quad i, piece g.  Row-major: row nc[f] of the segment, piece g of the step.
  unsigned vrow4[F], vrow6[F], vrow8[F];
  const unsigned vlane = (unsigned)(i * 64 + g * 16);
#pragma unroll
  for (int f = 0; f < F; ++f) {
    vrow4[f] = (unsigned)nc[f] * (unsigned)nblk4 * 16u + (unsigned)g * 16u;
    vrow6[f] = (unsigned)nc[f] * (unsigned)nblk6 * 16u + (unsigned)g * 16u;
    vrow8[f] = (unsigned)nc[f] * (unsigned)nblk8 * 16u + (unsigned)g * 16u;
  }
  const int wtile = (wg * F) >> 4, wj0 = (wg * F) & 15;
  auto request_step = [&](int r, auto buf_c, auto k_c) __attribute__((always_inline)) {
    constexpr int B = decltype(buf_c)::value, k = decltype(k_c)::value;
    {
      const int t = min(t_begin + r * S + k, total - 1);
      const int seg = t < s4.steps ? 0 : (t < s4.steps + s6.steps ? 1 : 2);
      const int q = seg == 0 ? t : (seg == 1 ? t - s4.steps : t - s4.steps - s6.steps);
      const uint8_t* pb = sel3p(seg, b4, b6, b8);
      if constexpr (WT) {
        const int nst = sel3(seg, nblk4, nblk6, nblk8) >> 2;
        const uint8_t* sb = pb + (((size_t)wtile * nst + q) * 16 + wj0) * 1024;
        if constexpr (F >= 1) load16_uncounted<0, true>(wq[B][k][0], sb, vlane);
        if constexpr (F >= 2) load16_uncounted<1024, true>(wq[B][k][F >= 2 ? 1 : 0], sb, vlane);
        if constexpr (F >= 4) {
          load16_uncounted<2048, true>(wq[B][k][F >= 4 ? 2 : 0], sb, vlane);
          load16_uncounted<3072, true>(wq[B][k][F >= 4 ? 3 : 0], sb, vlane);
        }
      } else {
        const uint8_t* sb = pb + (size_t)q * 64;
#pragma unroll
        for (int f = 0; f < F; ++f)
          load16_uncounted<0>(wq[B][k][f], sb, (unsigned)sel3(seg, (int)vrow4[f], (int)vrow6[f], (int)vrow8[f]));
      }
    }
  };
  auto request_round = [&](int r, auto buf_c) __attribute__((always_inline)) {
    request_step(r, buf_c, std::integral_constant<int, 0>{});
    request_step(r, buf_c, std::integral_constant<int, 1>{});
    request_step(r, buf_c, std::integral_constant<int, 2>{});
    request_step(r, buf_c, std::integral_constant<int, 3>{});
  };
  // ---- what is not a weight code, into LDS: requested first (measured: with the first round of weights ahead of
  // them the kernel is slower, by 2 % on tile-major and 7 % on row-major weights)
  copy_region(s4.a, M * nblk4 * 16, lds0 + L.x0, wave, lane);
  copy_region(s6.a, M * nblk6 * 24, lds0 + L.x1, wave, lane);
  copy_region(s8.a, M * nblk8 * 32, lds0 + L.x2, wave, lane);
  {
    const int palog = L.pa == 8 ? 3 : 4;
    // token scale pieces 0 ... pa - 1
    const unsigned pa_off = (unsigned)(lane & (L.pa - 1)) * 16u;
    if (s4.steps) copy_pieces(s4.sfa, s4.steps, palog, pa_off, lds0 + L.sfa0, wave, lane);
    if (s6.steps) copy_pieces(s6.sfa, s6.steps, palog, pa_off, lds0 + L.sfa1, wave, lane);
    if (s8.steps) copy_pieces(s8.sfa, s8.steps, palog, pa_off, lds0 + L.sfa2, wave, lane);
    if (s4.steps) copy_pieces(s4.sfb, s4.steps, PBLOG, sfb_piece_off + (unsigned)(sfb_katoms_mul * s4.steps) * 512u, lds0 + L.sfb0, wave, lane);
    if (s6.steps) copy_pieces(s6.sfb, s6.steps, PBLOG, sfb_piece_off + (unsigned)(sfb_katoms_mul * s6.steps) * 512u, lds0 + L.sfb1, wave, lane);
    if (s8.steps) copy_pieces(s8.sfb, s8.steps, PBLOG, sfb_piece_off + (unsigned)(sfb_katoms_mul * s8.steps) * 512u, lds0 + L.sfb2, wave, lane);
  }

  // The first two rounds: kAhead steps are requested up front, another one as each is used (a wave that requests more stands at its
  // requests while its first steps' codes are there).  Layer call from HBM, us, with both rounds requested and each waited for as a whole /
  // a window of 2 / 3 / 4 / 5 / 6 / 8 steps: N = 14336, K = 4096 (F = 4), M = 8 11.6 / 11.0 / 10.8 / 10.8 / 10.7 / 10.9 / 11.6, from the caches 10.0 / 10.0 /
  // 9.3 / 9.3 / 9.5 / 9.6 / 10.0; row-major, N = 18944, K = 3584 (F = 2), M = 16 17.0 / - / 16.85 / 16.3 / 16.4 / 16.3 / 16.7; N = K = 4096 (F = 1) 8.3, now 7.75.
  constexpr int kAhead = F == 4 ? 4 : (F == 2 ? 5 : 8);
  auto request_nth = [&](auto n_c) __attribute__((always_inline)) {
    constexpr int n = decltype(n_c)::value;
    request_step(n / S, std::integral_constant<int, n / S>{}, std::integral_constant<int, n % S>{});
  };
  // (the first round in one place for both cases: a register that is still to be filled must not have two loads meeting in it where branches join)
  static_assert(kAhead >= S, "the first round is requested up front");
  if (rounds > 0) for_each_step<0, S>(request_nth);
  if (rounds > 1) for_each_step<S, kAhead>(request_nth);

  // ---- the copies are older than all of them
  if (rounds > 1) wait_vmcnt<kAhead * F>();
  else if (rounds > 0) wait_vmcnt<S * F>();
  else wait_vmcnt<0>();
  asm volatile("s_barrier" ::: "memory");

  v4f acc[F];
#pragma unroll
  for (int f = 0; f < F; ++f) acc[f] = v4f{0.f, 0.f, 0.f, 0.f};
  // this lane's token (tokens past M: the last one again, never stored), and where its scale bytes sit in a step's pieces
  const int mc = min(i, M - 1), sx_off = mc * 16;
  const int pa16 = L.pa * 16;

  auto compute_step = [&](int r, auto buf_c, auto k_c) __attribute__((always_inline)) {
    constexpr int B = decltype(buf_c)::value, k = decltype(k_c)::value;
    {
      const int t = t_begin + r * S + k;
      if (t < t_end) {   // wave-uniform
        const int seg = t < s4.steps ? 0 : (t < s4.steps + s6.steps ? 1 : 2);
        const int q = seg == 0 ? t : (seg == 1 ? t - s4.steps : t - s4.steps - s6.steps);
        const uint8_t* sfa_l = lds + sel3(seg, L.sfa0, L.sfa1, L.sfa2) + q * pa16;
        const uint8_t* sfb_l = lds + sel3(seg, L.sfb0, L.sfb1, L.sfb2) + q * (PB * 16);
        const int s_x = sfa_l[sx_off + g];
        v8i wf[F];
        int s_w[F];
#pragma unroll
        for (int f = 0; f < F; ++f) {
          s_w[f] = sfb_l[piece[f] * 16 + slot[f] * 4 + g];
          const v4i w4 = wq[B][k][f];
          wf[f] = v8i{w4[0], w4[1], w4[2], w4[3], 0, 0, 0, 0};
        }
        if (seg == 0) {
          const v4i a4 = *reinterpret_cast<const v4i*>(lds + L.x0 + mc * (nblk4 * 16) + q * 64 + g * 16);
          const v8i xf = {a4[0], a4[1], a4[2], a4[3], 0, 0, 0, 0};
#pragma unroll
          for (int f = 0; f < F; ++f) acc[f] = decode_mfma<kFmtE2M1>(wf[f], xf, acc[f], s_w[f], s_x);
        } else if (seg == 1) {
          const v2i* p = reinterpret_cast<const v2i*>(lds + L.x1 + mc * (nblk6 * 24) + q * 96 + g * 24);
          const v2i a = p[0], b = p[1], c = p[2];
          const v8i xf = {a[0], a[1], b[0], b[1], c[0], c[1], 0, 0};
#pragma unroll
          for (int f = 0; f < F; ++f) acc[f] = decode_mfma<kFmtE3M2>(wf[f], xf, acc[f], s_w[f], s_x);
        } else {
          const uint8_t* p = lds + L.x2 + mc * (nblk8 * 32) + q * 128 + g * 16;
          const v4i a4 = *reinterpret_cast<const v4i*>(p), b4v = *reinterpret_cast<const v4i*>(p + 64);
          const v8i xf = {a4[0], a4[1], a4[2], a4[3], b4v[0], b4v[1], b4v[2], b4v[3]};
#pragma unroll
          for (int f = 0; f < F; ++f) acc[f] = decode_mfma<kFmtE4M3>(wf[f], xf, acc[f], s_w[f], s_x);
        }
      }
    }
  };
  auto compute_round = [&](int r, auto buf_c) __attribute__((always_inline)) {
    compute_step(r, buf_c, std::integral_constant<int, 0>{});
    compute_step(r, buf_c, std::integral_constant<int, 1>{});
    compute_step(r, buf_c, std::integral_constant<int, 2>{});
    compute_step(r, buf_c, std::integral_constant<int, 3>{});
  };
  // the registers of a round are tied to the wait that precedes their use
  auto settle = [&](auto buf_c, auto n_c) {
    constexpr int B = decltype(buf_c)::value;
    constexpr int NW = decltype(n_c)::value;
    wait_vmcnt<NW>();
#pragma unroll
    for (int k = 0; k < S; ++k)
#pragma unroll
      for (int f = 0; f < F; ++f) tie(wq[B][k][f]);
  };
  // The first two rounds are straight-line code, a window of requested steps (above); the loop behind them requests two whole rounds itself
  // and uses them: nothing is in flight across a loop edge (a register that an uncounted load is still to fill must not be
  // moved by the compiler, which a value carried around a loop may be).
  // Step n of kTotal; those up to n + kWin - 1 are requested.
  auto nth_step = [&](auto n_c, auto total_c) __attribute__((always_inline)) {
    constexpr int n = decltype(n_c)::value, kTotal = decltype(total_c)::value, kWin = kTotal > S ? kAhead : S;
    wait_vmcnt<(kWin - 1 < kTotal - 1 - n ? kWin - 1 : kTotal - 1 - n) * F>();
#pragma unroll
    for (int f = 0; f < F; ++f) tie(wq[n / S][n % S][f]);
    compute_step(n / S, std::integral_constant<int, n / S>{}, std::integral_constant<int, n % S>{});
    if constexpr (n + kWin < kTotal) request_nth(std::integral_constant<int, n + kWin>{});
  };
  if (rounds > 1) for_each_step<0, 2 * S>([&](auto n_c) __attribute__((always_inline)) { nth_step(n_c, std::integral_constant<int, 2 * S>{}); });
  else if (rounds > 0) for_each_step<0, S>([&](auto n_c) __attribute__((always_inline)) { nth_step(n_c, std::integral_constant<int, S>{}); });
  for (int r = 2; r < rounds; r += 2) {
    request_round(r, std::integral_constant<int, 0>{});
    if (r + 1 < rounds) {
      request_round(r + 1, std::integral_constant<int, 1>{});
      settle(std::integral_constant<int, 0>{}, std::integral_constant<int, S * F>{});
    } else {
      settle(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    }
    compute_round(r, std::integral_constant<int, 0>{});
    if (r + 1 < rounds) {
      settle(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
      compute_round(r + 1, std::integral_constant<int, 1>{});
    }
  }

  // ---- sum the four waves' partial tiles (D^T: lane holds token lane % 16, feature slots 4 * (lane / 16) + v of a group)
  float* partial = reinterpret_cast<float*>(lds + L.partial);
#pragma unroll
  for (int f = 0; f < F; ++f) *reinterpret_cast<v4f*>(partial + ((wave * F + f) * 64 + lane) * 4) = acc[f];
  __syncthreads();
  if (wave >= F) return;
  const int f = wave;
  v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 4; ++w) sum += *reinterpret_cast<const v4f*>(partial + ((w * F + f) * 64 + lane) * 4);
  if (i >= M) return;
  if constexpr (WT) {
    // feature slot e = 4 g + v of the block is row j + 32 (e % 8) + 16 (e / 8) of the tile
    const int bx = wg * F + f, row0 = (bx >> 4) * 256 + (bx & 15);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int e = 4 * g + v;
      store1(d, ep, i, row0 + 32 * (e & 7) + 16 * (e >> 3), sum[v]);
    }
  } else {
    // feature slots 4 g ... 4 g + 3 of the group are four consecutive rows
    const int per_group = 32 / PB, group = blockIdx.x / per_group, c0 = (blockIdx.x % per_group) * PB;
    const int e = 16 * f + 4 * g;
    store4(d, ep, i, group * 128 + c0 + e % PB + 32 * (e / PB), sum);
  }
}

// ---------------------------------------------------------------------------
// Token kernel: quantization and GEMM of a few tokens in one launch.
//
// For a token or two the quantizer is a launch of as many workgroups whose 2.5 us are latency, one memory round trip
// after the other, in front of a GEMM that waits for a round trip of its own.  Here every workgroup quantizes the tokens
// for itself, in LDS, while its first weights are on their way: x, the index (and the RMSNorm's weight) are copied to
// LDS, then the weight scales, then the first NS - 1 steps of weight codes of each ring; the tokens are gathered and
// quantized, their codes and scale bytes written to LDS, while the weights arrive.  The K loop is the skinny kernel's
// with one token group, its slots holding weight codes only.  The arithmetic is the quantizer's and the sums are added in the
// order of the decode and the skinny kernel: the same bits.  With RMSNorm the fp64 sum of squares is split over other lanes
// and waves than in the quantizer; its rounding to fp32 hides that unless the two sums, equal to about 2^-50, lie on two sides
// of a rounding boundary of fp32.
//
// What bounds it is latency: launch, first copies, LDS gathers (~0.5 us for every 8192 channels of the tokens), then the
// weights' arrival (counters, N = K = 4096, M = 1: waves waiting 66 % of their cycles, address unit busy 12 %, vector ALUs
// 12 %).  N = 4096, K = 4096, tile-major, in a graph, two launches -> one: M = 1 7.5 -> 6.0 us, 2 7.9 -> 6.4, 4 7.7 -> 7.5
// (8: 7.8 -> 10.0, not taken); N = 14336, M = 1 10.3 -> 8.0, 4 10.2 -> 9.3; with RMSNorm, N = 4096: M = 1 8.2 -> 7.1, 2
// 8.4 -> 8.0 (4: 8.4 -> 9.7, not taken).  A layer call of one token from Python: 9.1 -> 7.0 us.
// With shorter rings and whole steps two at a time (from HBM, one launch before and after): N = K = 4096, M = 1 6.2 -> 5.9, 2 6.6 -> 6.35, with
// RMSNorm 7.15 -> 6.9; N = K = 8192, M = 1 10.7 -> 9.9; N = 4096, K = 8192 9.1 -> 8.4; 200 drawn calls 1.035 times as fast in the mean.
// ---------------------------------------------------------------------------
constexpr int kTokenRows = 8;    // most tokens (a wave each in the RMSNorm)
constexpr int kTokenWaves = 8;   // all quantize; four of them also run the K loop
struct TokenLds {   // byte offsets behind the rings
  int x, idx, gamma;     // bf16 rows, index, RMSNorm weight
  int q0, q1, q2;        // codes per segment
  int sx0, sx1, sx2;     // their scale bytes: per step kTokenRows x 4
  int sw0, sw1, sw2;     // weight scale pieces: per step 4 F x 16
  int sums;              // RMSNorm: the waves' sums of squares
  int total;
};
// Slots per wave: 20 ... 64 KB of weight codes in flight per CU (see kSkinnySlots; with 12 / 8 / 5 of them, us: N = K = 4096 6.2, now 5.9; N = K =
// 8192 10.7, now 9.9; N = 14336, K = 4096 8.6, now 8.5)
template <int F>
constexpr int kTokenSlots = F == 1 ? 5 : (F == 2 ? 5 : 4);

// Codes and scale byte of half a block to LDS.
struct LdsHalf {
  uint8_t* q;    // of the block
  uint8_t* sf;
  int half;
  __device__ __forceinline__ void scale(int byte) const { *sf = (uint8_t)byte; }
  __device__ __forceinline__ void codes(v2u v) const { *reinterpret_cast<v2u*>(q + half * 8) = v; }
  __device__ __forceinline__ void codes(v3u v) const {
    unsigned* p = reinterpret_cast<unsigned*>(q + half * 12);
    p[0] = v[0]; p[1] = v[1]; p[2] = v[2];
  }
  __device__ __forceinline__ void codes(v4u v) const { *reinterpret_cast<v4u*>(q + half * 16) = v; }
};

__device__ __forceinline__ void lds_barrier() {   // this wave's LDS accesses are done, then every wave's
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int F, bool WT, bool NORM>
__global__ void __launch_bounds__(64 * kTokenWaves)
mixed_gemm_token_kernel(const uint8_t* __restrict__ x, const uint8_t* __restrict__ gamma, const uint8_t* __restrict__ idx,
                        float eps, int K, DecodeSeg s4, DecodeSeg s6, DecodeSeg s8, int M, int N, int steps_per_wave,
                        TokenLds L, Epilogue ep, uint16_t* __restrict__ d) {
  constexpr int NS = kTokenSlots<F>, kSlot = 1024 * F;
  constexpr int PB = 4 * F, PBLOG = F == 1 ? 2 : (F == 2 ? 3 : 4);
  // (four feature groups: 8.45 us one at a time, 8.6 in pairs; two on row-major weights: 80 calls from HBM / from the caches 1.6 % and 1.3 %
  // faster one at a time, N = 7936, K = 2048, M = 2 5.05 -> 4.9)
  constexpr bool kPairs = F == 1 || (F == 2 && WT);
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  // four waves share the K steps, as in the other kernels
  const uint8_t* const ring = lds + wave * (NS * kSlot);
  const unsigned ring0 = lds0 + (unsigned)wave * (NS * kSlot);
  const int t6 = s4.steps, t8 = s4.steps + s6.steps, total = t8 + s8.steps;
  const int t_begin = wave < 4 ? wave * steps_per_wave : total, t_end = min(total, t_begin + steps_per_wave);

  // ---- what everybody waits for first: tokens, index, RMSNorm weight, weight scales
  copy_region<kTokenWaves>(x, M * K * 2, lds0 + L.x, wave, lane);
  copy_region<kTokenWaves>(idx, K * 2, lds0 + L.idx, wave, lane);
  if constexpr (NORM) copy_region<kTokenWaves>(gamma, K * 2, lds0 + L.gamma, wave, lane);

  // ---- the workgroup's weight rows, as in the skinny kernel
  int wg = blockIdx.x;
  if constexpr (WT) {
    constexpr int kPer = 16 / F;
    if ((int)gridDim.x % (8 * kPer) == 0) {
      const int xcd = wg & 7, slot = wg >> 3;
      wg = ((slot / kPer) * 8 + xcd) * kPer + slot % kPer;
    }
  }
  constexpr int per_group = 32 / PB;
  const int tile = (wg * F) >> 4, j0 = (wg * F) & 15;                    // tile-major
  const int group = wg / per_group, c0 = (wg % per_group) * PB;          // row-major
  auto feature = [&](int f, int e) {
    if constexpr (WT) return tile * 256 + j0 + f + 32 * (e & 7) + 16 * (e >> 3);
    else return group * 128 + c0 + (16 * f + e) % PB + 32 * ((16 * f + e) / PB);
  };
  int sw_off[F], wrow[F];
#pragma unroll
  for (int f = 0; f < F; ++f) {
    if constexpr (WT) sw_off[f] = (((i & 7) >> 2) * 2 * F + (i >> 3) * F + f) * 16 + (i & 3) * 4 + g;
    else sw_off[f] = ((16 * f + i) % PB) * 16 + ((16 * f + i) / PB) * 4 + g;
    wrow[f] = min(feature(f, lane >> 2), N - 1);   // rows past N: read again, never stored
  }
  {
    const int pl = lane % PB;
    const unsigned piece = WT ? (unsigned)(j0 + pl % F + 16 * ((pl / F) & 1)) * 16u : (unsigned)(c0 + pl) * 16u;
    const unsigned mul = WT ? (unsigned)(tile * 2 + pl / (2 * F)) : (unsigned)group;
    if (s4.steps) copy_pieces<kTokenWaves>(s4.sfb, s4.steps, PBLOG, piece + mul * (unsigned)s4.steps * 512u, lds0 + L.sw0, wave, lane);
    if (s6.steps) copy_pieces<kTokenWaves>(s6.sfb, s6.steps, PBLOG, piece + mul * (unsigned)s6.steps * 512u, lds0 + L.sw1, wave, lane);
    if (s8.steps) copy_pieces<kTokenWaves>(s8.sfb, s8.steps, PBLOG, piece + mul * (unsigned)s8.steps * 512u, lds0 + L.sw2, wave, lane);
  }

  // ---- the first steps of weight codes
  const int wpos = (lane & 3) ^ ((lane >> 4) & 3);   // the 16-byte piece of its row that this lane copies
  auto request = [&](int t, unsigned slot) __attribute__((always_inline)) {
    if (t >= t_end) return;
    const int seg = t < t6 ? 0 : (t < t8 ? 1 : 2), q = t - sel3(seg, 0, t6, t8);
    const uint8_t* b = sel3p(seg, s4.b, s6.b, s8.b);
    const int nblk = sel3(seg, s4.nblk, s6.nblk, s8.nblk), whole = nblk >> 2, left = min(nblk - 4 * q, 4);
    const unsigned wp = (unsigned)min(wpos, left - 1) * 16u;
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const unsigned at = slot + 1024u * f;
      if constexpr (WT) {
        if (q < whole) dma16_at(b + (((size_t)tile * whole + q) * 16 + j0 + f) * 1024, (unsigned)(lane >> 2) * 64u + wp, at);
        else dma16_at(b + (size_t)(N >> 8) * whole * 16384, (unsigned)wrow[f] * (unsigned)(nblk & 3) * 16u + wp, at);
      } else {
        dma16_at(b + (size_t)q * 64, (unsigned)wrow[f] * (unsigned)nblk * 16u + wp, at);
      }
    }
  };
#pragma unroll
  for (int k = 0; k < NS - 1; ++k) request(t_begin + k, ring0 + k * kSlot);
  wait_steps<F, NS - 1>(min(NS - 1, t_end - t_begin));   // everything older has landed
  lds_barrier();

  // ---- RMSNorm of the tokens, in place (see the quantizer); the waves are dealt to the tokens
  if constexpr (NORM) {
    double* sums = reinterpret_cast<double*>(lds + L.sums);
    // token wave >> shift, shared by `of` waves of which this is the rank-th
    const int shift = M == 1 ? 3 : (M == 2 ? 2 : (M <= 4 ? 1 : 0)), of = 1 << shift;
    const int m = wave >> shift, rank = wave & (of - 1), pieces = m < M ? K >> 3 : 0;
    uint8_t* row = lds + L.x + m * K * 2;
    double part[4] = {0.0, 0.0, 0.0, 0.0};
    for (int p = rank * 64 + lane; p < pieces; p += of * 64) {
      const v4u a = *reinterpret_cast<const v4u*>(row + p * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double lo = (double)__uint_as_float(a[e] << 16), hi = (double)__uint_as_float(a[e] & 0xffff0000u);
        part[e] = __builtin_fma(lo, lo, part[e]);
        part[e] = __builtin_fma(hi, hi, part[e]);
      }
    }
    const double ss = wave_sum((part[0] + part[1]) + (part[2] + part[3]));
    if (lane == 0) sums[wave] = ss;
    lds_barrier();
    double tot = 0.0;
    for (int w = 0; w < of; ++w) tot += sums[m * of + w];
    const float r = rms_scale(tot, K, 1.0 / (double)K, eps);
    for (int p = rank * 64 + lane; p < pieces; p += of * 64) {
      v4u* at = reinterpret_cast<v4u*>(row + p * 16);
      const v4u gm = *reinterpret_cast<const v4u*>(lds + L.gamma + p * 16);
      v4u a = *at;
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = rms_apply(a[e], gm[e], r);
      *at = a;
    }
    lds_barrier();
  }

  // ---- quantization: two lanes per block of 32 (a pair is always both inside or both outside)
  const int halves = K >> 4;
  for (int m = 0, h = tid; ; h += 64 * kTokenWaves) {
    while (h >= halves && m < M) {   // on to the next token
      h -= halves;
      ++m;
    }
    if (m >= M) break;
    const int b = h >> 1, half = h & 1;
    const int seg = b < s4.nblk ? 0 : (b < s4.nblk + s6.nblk ? 1 : 2);
    const int j = b - sel3(seg, 0, s4.nblk, s4.nblk + s6.nblk);
    const int fmt = sel3(seg, kFmtE2M1, kFmtE3M2, kFmtE4M3), bytes = sel3(seg, 16, 24, 32);
    uint8_t* q = lds + sel3(seg, L.q0 + m * s4.nblk * 16, L.q1 + m * s6.nblk * 24, L.q2 + m * s8.nblk * 32) + j * bytes;
    uint8_t* sf = lds + sel3(seg, L.sx0, L.sx1, L.sx2) + (j >> 2) * (4 * kTokenRows) + m * 4 + (j & 3);
    const v4u i0 = *reinterpret_cast<const v4u*>(lds + L.idx + h * 32), i1 = *reinterpret_cast<const v4u*>(lds + L.idx + h * 32 + 16);
    int at[16];   // an entry outside [0, K) reads channel K - 1
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const unsigned w = e < 8 ? i0[e >> 1] : i1[(e - 8) >> 1];
      at[e] = L.x + m * K * 2 + (int)min((e & 1) ? w >> 16 : w & 0xffffu, (unsigned)(K - 1)) * 2;
    }
    float f[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) f[e] = __uint_as_float((unsigned)*reinterpret_cast<const uint16_t*>(lds + at[e]) << 16);
    quantize_half(f, fmt, half, LdsHalf{q, sf, half});
  }
  lds_barrier();

  // ---- the K loop
  v4f acc[F];
#pragma unroll
  for (int f = 0; f < F; ++f) acc[f] = v4f{0.f, 0.f, 0.f, 0.f};
  const int mc = min(i, M - 1);   // tokens past M: the last one again, never stored
  int t = t_begin, slot = 0;
  struct Fragments { v4i w[F]; v8i x; int s_w[F], s_x; };
  // the wave's steps of one segment, whole ones two at a time as in the skinny kernel
  auto run = [&](auto fmt_c, const DecodeSeg& s, int codes, int sfx, int sfw, int t_first, int t_next) __attribute__((always_inline)) {
    constexpr int FMT = decltype(fmt_c)::value;
    const int last = min(t_next, t_end);
    if (t >= last) return;
    const int whole_end = min(last, t_first + (s.nblk >> 2));
    const uint8_t* row = lds + codes + mc * (s.nblk * Frag<FMT>::kBytes) + g * (FMT == kFmtE3M2 ? 24 : 16);
    const uint8_t* sx = lds + sfx + mc * 4 + g;
    const uint8_t* sw = lds + sfw;
    auto read = [&](Fragments& r, const uint8_t* sl, int q) __attribute__((always_inline)) {
      r.s_x = sx[q * (4 * kTokenRows)];
#pragma unroll
      for (int f = 0; f < F; ++f) {
        r.s_w[f] = sw[q * (PB * 16) + sw_off[f]];
        r.w[f] = *reinterpret_cast<const v4i*>(sl + 1024 * f + i * 64 + (g ^ ((i >> 2) & 3)) * 16);
      }
      if constexpr (FMT == kFmtE2M1) {
        const v4i a = *reinterpret_cast<const v4i*>(row + q * 64);
        r.x = v8i{a[0], a[1], a[2], a[3], 0, 0, 0, 0};
      } else if constexpr (FMT == kFmtE3M2) {
        const v2i* p = reinterpret_cast<const v2i*>(row + q * 96);
        const v2i a = p[0], b = p[1], e = p[2];
        r.x = v8i{a[0], a[1], b[0], b[1], e[0], e[1], 0, 0};
      } else {
        const v4i a = *reinterpret_cast<const v4i*>(row + q * 128);
        const v4i b = *reinterpret_cast<const v4i*>(row + q * 128 + 64);
        r.x = v8i{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      }
    };
    auto multiply = [&](const Fragments& r) __attribute__((always_inline)) {
#pragma unroll
      for (int f = 0; f < F; ++f)
        acc[f] = decode_mfma<FMT>(v8i{r.w[f][0], r.w[f][1], r.w[f][2], r.w[f][3], 0, 0, 0, 0}, r.x, acc[f], r.s_w[f], r.s_x);
    };
    // the last steps at once with one and two feature groups, else each by itself (400 calls of up to 8 tokens, K < 2600 and up to 18944, at once
    // over each by itself from the caches / from HBM: one and two groups 0.5 ... 2.9 % / 0 ... 1.8 % faster, four 1.3 % and 0.3 % faster / 1.4 % and 0.8 %
    // slower)
    auto wait_for = [&](auto steps_c) __attribute__((always_inline)) {
      constexpr int kSteps = decltype(steps_c)::value;
      if (t + NS - 1 < t_end) wait_vmcnt<(NS - kSteps) * F>();
      else if constexpr (F < 4) wait_vmcnt<0>();
      else wait_steps<F, NS - 1 - kSteps>(t_end - kSteps - t);
    };
    while (t < last) {
      const uint8_t* sl = ring + slot * kSlot;
      const unsigned this_slot = ring0 + (unsigned)slot * kSlot;
      request(t + NS - 1, ring0 + (unsigned)(slot == 0 ? NS - 1 : slot - 1) * kSlot);
      slot = slot == NS - 1 ? 0 : slot + 1;
      const int q = t - t_first;
      if (kPairs && t + 1 < whole_end) {
        wait_for(std::integral_constant<int, 2>{});
        Fragments r0, r1;
        read(r0, sl, q);
        read(r1, ring + slot * kSlot, q + 1);
        // the weights are in registers before a later request may fill these slots again
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        request(t + NS, this_slot);
        multiply(r0);
        multiply(r1);
        slot = slot == NS - 1 ? 0 : slot + 1;
        t += 2;
        continue;
      }
      wait_for(std::integral_constant<int, 1>{});
      const int left = s.nblk - 4 * q;
      Fragments r;
      read(r, sl, q);
      if (left < 4) {   // wave-uniform: the segment's last, partial step; what lies past its end is zero
        const bool ok = g < left, lo_ok = FMT == kFmtE4M3 ? (g >> 1) < left : ok, hi_ok = FMT == kFmtE4M3 ? 2 + (g >> 1) < left : ok;
        r.s_x = ok ? r.s_x : 127;
#pragma unroll
        for (int f = 0; f < F; ++f) {
          r.s_w[f] = ok ? r.s_w[f] : 127;
#pragma unroll
          for (int e = 0; e < 4; ++e) r.w[f][e] = ok ? r.w[f][e] : 0;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          r.x[e] = lo_ok ? r.x[e] : 0;
          r.x[4 + e] = hi_ok ? r.x[4 + e] : 0;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      multiply(r);
      ++t;
    }
  };
  run(std::integral_constant<int, kFmtE2M1>{}, s4, L.q0, L.sx0, L.sw0, 0, t6);
  run(std::integral_constant<int, kFmtE3M2>{}, s6, L.q1, L.sx1, L.sw1, t6, t8);
  run(std::integral_constant<int, kFmtE4M3>{}, s8, L.q2, L.sx2, L.sw2, t8, total);

  // ---- sum the four waves' partial tiles, in the rings' place
  lds_barrier();
  float* partial = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int f = 0; f < F; ++f)
    if (wave < 4) *reinterpret_cast<v4f*>(partial + ((wave * F + f) * 64 + lane) * 4) = acc[f];
  __syncthreads();
  if (wave >= F || i >= M) return;
  const int f = wave;
  v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 4; ++w) sum += *reinterpret_cast<const v4f*>(partial + ((w * F + f) * 64 + lane) * 4);
  if constexpr (WT) {
#pragma unroll
    for (int v = 0; v < 4; ++v) store1(d, ep, i, feature(f, 4 * g + v), sum[v]);
  } else {
    store4(d, ep, i, feature(f, 4 * g), sum);
  }
}

static int round_up_1k(int v) { return (v + 1023) & ~1023; }

// The decode kernel takes whole 128-wide steps in every segment and an LDS image of at most 76 KB.
constexpr int kDecodeLds = 76 * 1024;
static bool decode_lds_plan(const DecodeSeg& d4, const DecodeSeg& d6, const DecodeSeg& d8, int M, int F, DecodeLds* L) {
  int pos = 0;
  auto take = [&](int bytes) { const int at = pos; pos += round_up_1k(bytes); return at; };
  L->pa = M <= 8 ? 8 : 16;
  L->x0 = take(M * d4.nblk * 16); L->x1 = take(M * d6.nblk * 24); L->x2 = take(M * d8.nblk * 32);
  L->sfa0 = take(d4.steps * L->pa * 16); L->sfa1 = take(d6.steps * L->pa * 16); L->sfa2 = take(d8.steps * L->pa * 16);
  L->sfb0 = take(d4.steps * F * 64); L->sfb1 = take(d6.steps * F * 64); L->sfb2 = take(d8.steps * F * 64);
  L->partial = pos;
  pos += 4 * F * 1024;
  L->total = pos;
  return pos <= kDecodeLds;
}

// Token groups (g) and feature groups (f) of 16 per workgroup of the skinny kernel, and its launch time in microseconds:
// the pair with the lowest estimate.  A workgroup takes ~2.3 us to fill and drain its pipeline plus the table's nanoseconds per
// K step; a further round of workgroups costs more than the first (fitted).  A round is a workgroup per CU, also for (1, 1) and
// (1, 2), of which three and two fit a CU's LDS: side by side they share its requests, and the form with half as many workgroups is
// faster (M = 16, K = 4096, us from the caches / from HBM, two workgroups of (1, 1) per CU against one of (1, 2): N = 8192 tile-major 6.4
// against 5.4 / 8.15 against 6.6, row-major 6.45 against 5.6 / 8.3 against 7.4; two of (1, 2) against one of (1, 4), N = 12288 7.9 against 7.5 / 10.3
// against 8.9, row-major 8.4 against 8.2 / 11.3 against 10.2).
// Row-major weights have a column of their own (a weight copy touches 16 half lines there, 8 lines on tile-major ones): the
// smallest forms are cheaper than on tile-major weights, the two largest dearer, which changes their order.  Two and four
// token groups with one feature group are not among the forms: half the token groups with twice the feature groups are never
// more workgroups, and cheaper (83 against 77 and 99 against 86 ns on tile-major weights, 69 / 62 and 96 / 89 on row-major).
// Estimate against measurement, with the weights in the caches / from HBM (rotating over 1.3 GB), us:
//   tile-major, N = 4096, K = 14336: M = 16 10.9 against 9.3 / 11.6, 128 15.7 against 17.1 / 22.7; N = K = 5120: M = 8 6.5 against
//     5.75 / 6.7; N = 2560, K = 5120, M = 128 7.8 against 8.6 / 11.0
//   row-major, N = 4096, K = 14336: M = 16 8.5 against 8.95 / 12.2, 128 18.4 against 20.2 / 25.2; N = K = 5120: M = 8 5.8 against
//     5.3 / 7.5
// Eight feature groups are for 64 to 128 features per CU and up to 16 tokens, where four need a second round (from HBM, M = 16,
// tile-major / row-major weights, us): N = 20480, K = 5120 19.3 -> 16.3 / 23.6 -> 20.6, N = 28672, K = 5120 22.0 -> 17.1 / 25.9 -> 22.6, N =
// 18944, K = 3584 15.7 -> 11.6.  Up to 64 features per CU they are slower (N = 16384, K = 5120 15.2 against 12.3), and so they are
// with two token groups (M = 32, N = 24576, K = 8192 21.4 against 19.1 on small tiles).
// Over 1511 calls of 17 to 255 tokens (N 256 ... 28672, K 1024 ... 18944) the form taken, whole tiles included, is in the
// mean 1.2 / 3.0 % (row-major) and 2.0 / 3.2 % (tile-major) slower than the best one, 22 / 60 % and 27 / 40 % at most; with the
// tile-major figures row-major weights were at 3.0 / 5.2 and 68 / 77 %.
// On tile-major weights (2, 2) and (4, 2) give way to half the tokens and twice the features wherever those are as many workgroups: M = 56, N =
// 3584, K = 8192 (1, 4) against (2, 2) 8.6 / 11.2 against 8.6 / 11.6; M = 64, N = K = 4096 6.35 / 7.7 against 6.0 / 8.1; M = 128, N = K = 4096 (2, 4)
// against (4, 2) 7.8 / 9.7 against 8.3 / 10.2, K = 14336 17.1 / 22.7 against 19.1 / 24.5.  The estimate is the same for both.
struct SkinnyPlan { int g, f; double us; };
static SkinnyPlan skinny_plan(int M, int N, int steps, int cus, bool w_tiled) {
  static const struct { int g, f; double ns[2]; } kForms[] = {   // row-major, tile-major weights
      {1, 1, {46, 67}}, {1, 2, {62, 77}}, {1, 4, {104, 102}}, {2, 2, {89, 86}}, {2, 4, {145, 117}}, {4, 2, {134, 110}}, {1, 8, {230, 225}}};
  SkinnyPlan best = {0, 0, 0.0};
  for (const auto& k : kForms) {
    if (k.f == 8 && M > 16) continue;
    const int across = w_tiled ? ceil_div(N, 16 * k.f) : ceil_div(N, 128) * (8 / k.f);
    const int rounds = (int)(((int64_t)across * ceil_div(M, 16 * k.g) + cus - 1) / cus);
    const double us = 1.0 + rounds * (2.3 + steps * k.ns[w_tiled] * 1e-3) + 1.5 * (rounds - 1);
    if (best.g == 0 || us < best.us) best = {k.g, k.f, us};
  }
  if (w_tiled && best.g >= 2 && best.f == 2 && ceil_div(M, 8 * best.g) == 2 * ceil_div(M, 16 * best.g)) best = {best.g / 2, 4, best.us};
  return best;
}

// The decode kernel, which brings the tokens' codes and all scales into LDS once per workgroup, for up to 16 tokens and
// whole 128-wide steps: its feature groups of 16 per workgroup, or 0 where another kernel is taken.
// Against the skinny kernel on tile-major weights, K = 4096, from the caches / from HBM (layers of 120 and of 700 MB in turn, us):
//   N = 4096 (1 feature group per workgroup): M = 4 5.3 against 5.5 / 5.5 against 5.9, 16 (skinny) 5.5 against 5.3 / 5.8 against 6.6;
//   N = 14336 (4): M = 8 8.9 against 8.6 / 8.7 against 9.4, 16 9.3 against 8.8 / 9.2 against 10.1;
//   N = 28672 (4, two per CU; skinny with 8): M = 4 12.4 against 12.1 / 14.0 against 14.2, 16 13.3 against 13.3 / 15.3 against 14.2;
//   K = 8192, M = 4: N = 4096 8.6 against 7.7 / 8.7 against 8.1, 14336 15.6 against 13.1 / 14.5 against 14.9;
//   N = 18944, M = 16: K = 1024 7.8 against 7.2 / 7.2 against 6.7, 2048 8.9 against 8.8 / 8.8 against 8.7 (N = 28672: 8.7 against
//     9.5 / 9.1 against 9.6), 2560 12.0 against 9.7 / 12.1 against 9.7;  N = 36864, K = 3584, M = 16 18.7 against 20.9 / 19.0 against 23.1.
// (Both sides before the skinny kernel's shorter rings and this kernel's window of requested steps.  With them, layer calls from HBM / from the
// caches, skinny against this kernel, M = 16, K = 4096: N = 4096 8.5 against 8.1 / 8.0 against 8.5 us, 6144 9.7 against 8.9 / 8.4 against 8.8, 8192
// 10.0 against 9.1 / 8.5 against 8.9; the four projections of a decoder layer, 116 MB in a graph, 53.6 with the rule as it is, 55.9 with this
// kernel for up to 16 tokens on 4096 and 6144 features.)
// So: four feature groups (two such workgroups fit a CU), or one round of workgroups and at most 8 tokens; up to 32 K steps, which are
// the two rounds per wave that have a window of requests (the loop behind them starts with nothing in flight; M = 4, this kernel against
// the skinny one from the caches / from HBM, 32 and 36 steps: N = 4096 5.0 against 4.7 / 5.05 against 5.4 and 6.2 against 4.85 / 6.2 against 5.8, N =
// 14336 7.3 against 7.7 / 7.7 against 8.5 and 9.5 against 8.3 / 9.9 against 9.3); up to 16 where the skinny kernel has eight feature groups; above 128
// features per CU, where that needs two rounds, always.
// On row-major weights the skinny kernel is ahead or level up to 64 features per CU (N = 4096, K = 4096, M = 1: 5.1 against 5.6 / 5.4
// against 5.7; N = 14336, M = 16: 8.6 against 9.3 / 11.1 against 10.7), then needs eight feature groups or a second round, where two
// workgroups of this kernel with two feature groups fit a CU: N = 18944, M = 16: K = 2048 8.0 against 7.9 / 8.8 against 9.6, K = 3584
// 11.9 against 10.6 / 13.6 against 14.9, K = 4096 - / 14.0 against 16.1.
// The whole-tile kernel was slower than the form taken here at every shape measured (N = 28672, K = 2048: 11.4 against 8.8).
// (a segment's weight codes below 4 GB: the kernel addresses them with 32-bit per-lane offsets)
static int decode_plan(const DecodeSeg& d4, const DecodeSeg& d6, const DecodeSeg& d8, int M, int N, bool w_tiled, int cus,
                       DecodeLds* L) {
  const size_t widest = (size_t)(d4.nblk > d6.nblk ? (d4.nblk > d8.nblk ? d4.nblk : d8.nblk) : (d6.nblk > d8.nblk ? d6.nblk : d8.nblk));
  if (M > 16 || widest == 0 || ((d4.nblk | d6.nblk | d8.nblk) & 3) != 0 || (size_t)N * widest * 16 >= ((size_t)1 << 32)) return 0;
  int f = 2;
  if (w_tiled) {
    const int steps = d4.steps + d6.steps + d8.steps;
    f = ceil_div(N, 64) >= cus * 3 / 4 ? 4 : (ceil_div(N, 32) >= cus ? 2 : 1);
    if (f < 4 && (M > 8 || ceil_div(N, 16 * f) > cus)) return 0;
    if (ceil_div(N, 128) <= cus && steps > (ceil_div(N, 64) <= cus ? 32 : 16)) return 0;
  } else if (ceil_div(N, 128) * 2 <= cus) {
    return 0;
  }
  return decode_lds_plan(d4, d6, d8, M, f, L) ? f : 0;
}

hipError_t launch_decode(const DecodeSeg& d4, const DecodeSeg& d6, const DecodeSeg& d8, int M, int N, bool w_tiled, int f,
                         const DecodeLds& L, Epilogue ep, uint16_t* d, hipStream_t stream) {
  typedef void (*kernel_t)(DecodeSeg, DecodeSeg, DecodeSeg, int, int, int, DecodeLds, Epilogue, uint16_t*);
  const kernel_t kernel = !w_tiled ? mixed_gemm_decode_kernel<2, false> : (f == 4 ? mixed_gemm_decode_kernel<4, true> :
                          (f == 2 ? mixed_gemm_decode_kernel<2, true> : mixed_gemm_decode_kernel<1, true>));
  // row-major: per group of 128 rows 8 / F workgroups (the last group whole, rows past N clamped and not stored)
  const dim3 grid(w_tiled ? ceil_div(N, 16 * f) : ceil_div(N, 128) * (8 / f));
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kDecodeLds); e != hipSuccess) return e;
  const int total = d4.steps + d6.steps + d8.steps;
  hipLaunchKernelGGL(kernel, grid, dim3(256), (size_t)L.total, stream, d4, d6, d8, M, N, (total + 3) / 4, L, ep, d);
  return hipGetLastError();
}

hipError_t launch_skinny(const DecodeSeg& d4, const DecodeSeg& d6, const DecodeSeg& d8, int M, int N, bool w_tiled,
                         const SkinnyPlan& plan, Epilogue ep, uint16_t* d, hipStream_t stream) {
  const int total = d4.steps + d6.steps + d8.steps;
  const TileOrder order = tile_runs(w_tiled ? ceil_div(N, 16 * plan.f) : ceil_div(N, 128) * (8 / plan.f), ceil_div(M, 16 * plan.g));
  auto launch = [&](auto g_c, auto f_c) {
    constexpr int G = decltype(g_c)::value, F = decltype(f_c)::value;
    constexpr int kLds = 4 * kSkinnySlots<G, F> * kSkinnySlot<G, F>;
    const bool once = (total + 3) / 4 < kSkinnySlots<G, F>;
    const auto kernel = w_tiled ? (once ? mixed_gemm_skinny_kernel<G, F, true, true> : mixed_gemm_skinny_kernel<G, F, true, false>)
                                : (once ? mixed_gemm_skinny_kernel<G, F, false, true> : mixed_gemm_skinny_kernel<G, F, false, false>);
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds); e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(order.grid_x, grid_rows(order)), dim3(256), kLds, stream, d4, d6, d8, M, N, (total + 3) / 4, order, ep, d);
    return hipGetLastError();
  };
  const std::integral_constant<int, 1> one;
  const std::integral_constant<int, 2> two;
  const std::integral_constant<int, 4> four;
  const std::integral_constant<int, 8> eight;
  if (plan.g == 4) return launch(four, two);
  if (plan.g == 2) return plan.f == 4 ? launch(two, four) : launch(two, two);
  return plan.f == 8 ? launch(one, eight) : plan.f == 4 ? launch(one, four) : (plan.f == 2 ? launch(one, two) : launch(one, one));
}

}  // namespace

// 256 x 256 tiles, one workgroup per CU (mixed_gemm_256.hip)
bool mixed_gemm_256_supported(int M, int N, int KN, int KS, int KO);
hipError_t launch_mixed_gemm_256(const uint8_t* an, const uint8_t* bn, const uint8_t* as_, const uint8_t* bs,
                                 const uint8_t* ao, const uint8_t* bo, const uint8_t* sfan, const uint8_t* sfbn,
                                 const uint8_t* sfas, const uint8_t* sfbs, const uint8_t* sfao, const uint8_t* sfbo,
                                 int m_store, int a_rows, int a_staged, int N, int KN, int KS, int KO, bool w_tiled, Epilogue ep,
                                 void* d, hipStream_t stream);

// tiles of 64 or 128 features x 64 or 128 tokens (mixed_gemm_tile.hip)
struct TilePlanChoice { int tf, tt; double us; };
TilePlanChoice mixed_gemm_tile_plan(int M, int N, int KN, int KS, int KO, int cus);
hipError_t launch_mixed_gemm_tile(const uint8_t* an, const uint8_t* bn, const uint8_t* as_, const uint8_t* bs,
                                  const uint8_t* ao, const uint8_t* bo, const uint8_t* sfan, const uint8_t* sfbn,
                                  const uint8_t* sfas, const uint8_t* sfbs, const uint8_t* sfao, const uint8_t* sfbo,
                                  int m_store, int a_rows, int a_staged, int N, int KN, int KS, int KO, bool w_tiled, const TilePlanChoice& choice,
                                  Epilogue ep, void* d, hipStream_t stream);

// Rough launch time of the whole-tile kernel in microseconds for fewer than 256 tokens, only to choose between the kernels: as
// 256 x 128 tiles when that is at most one round (fitted to 771 calls on tile-major weights, rms error 8 %), else as 256 x 256.
// What the blocks past whole stages, the hand-over between three segments and an E3M2 segment shorter than its pipeline cost is
// counted: with 4.5 us for the last (K = 1024: N = 24576, M = 64 was 12.9 us here, and is 6.4 on small tiles; not counted for more than
// cus / 2 whole tiles).
static bool short_middle(int KN, int KS, int KO) { return KN > 0 && KO > 0 && KS > 0 && KS < 384; }
static double pipelined_us(int M, int N, int stages, int KN, int KS, int KO, int cus) {
  const int whole = ceil_div(M, 256) * ceil_div(N, 256), halves = ceil_div(M, 128) * ceil_div(N, 256);
  if (whole > cus / 2) return (double)ceil_div(whole, cus) * (stages * 0.95 + 3.0);
  return 1.9 + stages * (0.342 + 0.28 * fmin(1.0, (double)halves / cus)) + ((KN | KS | KO) % 128 != 0 ? 1.0 : 0.0) +
         (KN > 0 && KS > 0 && KO > 0 ? 2.0 : 0.0) + (short_middle(KN, KS, KO) ? 4.5 : 0.0);
}

// The same on tile-major weights for 256 tokens and more, fitted to 184 measured calls (rms error 7 %): half tiles (at most cus / 2
// whole ones) or rounds of whole tiles, of which a last one on at most half of the CUs counts 0.62; microseconds per stage, per
// MB of results, and what the blocks past whole stages cost.
static double whole_tiles_us(int M, int N, int stages, int KN, int KS, int KO, int cus) {
  const bool rest = (KN | KS | KO) % 128 != 0, three_segments = KN > 0 && KS > 0 && KO > 0;
  const int whole = ceil_div(M, 256) * ceil_div(N, 256), halves = ceil_div(M, 128) * ceil_div(N, 256);
  const double mb = 2e-6 * M * N;
  if (whole <= cus / 2) return 3.8 + stages * (0.346 + 0.084 * fmin(1.0, (double)halves / cus)) + 0.26 * mb + (rest ? 2.0 : 0.0) + (short_middle(KN, KS, KO) ? 4.5 : 0.0);
  const int full = whole / cus, left = whole % cus;
  const double rounds = full + (left == 0 ? 0.0 : (left <= cus / 2 && full > 0 && three_segments ? 0.62 : 1.0));
  return fmax(1.4 + rounds * (stages * 0.741 - 7.0 + (rest ? 2.5 : 0.0)) + 0.63 * mb, rounds * stages * 0.6);
}

// The kernel a problem runs on.  A function of the shape, the weights' layout and the number of CUs alone.
enum class GemmKernel { kNone, kDecode, kSkinny, kTile, kWhole };
struct GemmChoice {
  GemmKernel kernel;
  int decode_f;          // kDecode: feature groups of 16 per workgroup
  DecodeLds lds;         //   and the LDS image
  SkinnyPlan skinny;     // kSkinny
  TilePlanChoice tile;   // kTile
};

static GemmChoice choose_gemm(const DecodeSeg& d4, const DecodeSeg& d6, const DecodeSeg& d8, int M, int N, int KN, int KS, int KO,
                              bool w_tiled, int cus) {
  GemmChoice c = {};
  if (M == 0 || N == 0) return c;
  const int m_pad = (M + 255) / 256 * 256;
  const bool whole_tiles = mixed_gemm_256_supported(m_pad, N, KN, KS, KO);
  const int steps = d4.steps + d6.steps + d8.steps;
  // (the skinny kernel addresses a segment's row-major weight codes with 32-bit offsets)
  const int widest = KN > KS ? (KN > KO ? KN : KO) : (KS > KO ? KS : KO);
  const bool few = M < 256 && KN + KS + KO > 0, skinny_ok = few && (w_tiled || (size_t)N * (size_t)(widest / 2) < ((size_t)1 << 32));
  if (few) {
    c.decode_f = decode_plan(d4, d6, d8, M, N, w_tiled, cus, &c.lds);
    if (c.decode_f != 0) {
      c.kernel = GemmKernel::kDecode;
      return c;
    }
  }
  // What no other kernel takes, whatever the number of tokens, goes to small tiles; so does what they are estimated to be the
  // fastest for by a margin (the estimates of both sides are off by 10 %), above 16 tokens.  Both weight layouts go the same way
  // there (they give the same bits): the estimates compared are those on tile-major weights.
  // (128 tokens, N = K = 4096, the nearest of the estimates: 9.6 against 8.2 us on small tiles with the weights in the caches, 10.8
  // against 10.9 from HBM.)
  // The margins: 5 %; 0.6 us more against the skinny kernel up to 9 steps, where the launch ramps are all there is (from HBM, small tile
  // against skinny: M = 18, N = 2560, K = 1024 5.0 against 3.3 us, M = 21, N = 8360 5.4 against 4.6); 7 % against whole tiles below 256
  // tokens where the small ones need a second round (M = 171, N = 20480, K = 11008, row-major 48.6 against 44.3).
  // Against the choice between the other kernels alone, 4882 drawn calls of 17 ... 255 tokens: 1.22 times as fast in the mean with the
  // weights in the caches, 1.17 from HBM, 13 of them slower by more than 3 %; 2297 of 256 ... 3000 tokens: 1.22 and 1.24, 4 slower.  Most
  // of these are row-major weights of 100 MB and more in a tile or two of tokens (M = 23, N = 17984, K = 13824 43.6 against 41.8), at worst N =
  // 16440, K = 18944 as MXFP4 and MXFP8, M = 19 67 against 52 us; the mean over their neighbours is 1.05.
  c.tile = mixed_gemm_tile_plan(M, N, KN, KS, KO, cus);
  const SkinnyPlan skinny_t = few ? skinny_plan(M, N, steps, cus, true) : SkinnyPlan{0, 0, 0.0};
  const double whole_us = few ? pipelined_us(M, N, steps, KN, KS, KO, cus) : whole_tiles_us(M, N, steps, KN, KS, KO, cus);
  const bool second_round = (int64_t)ceil_div(N, c.tile.tf) * ceil_div(M, c.tile.tt) > cus;
  const bool before_whole = c.tile.us < (few && second_round ? 0.93 : 0.95) * whole_us;
  const bool before_skinny = c.tile.us + (steps <= 9 ? 0.6 : 0.0) < 0.95 * skinny_t.us;
  const bool fastest = few ? M > 16 && before_skinny && (!whole_tiles || before_whole) : before_whole;
  if ((!whole_tiles && !skinny_ok) || fastest) {
    c.kernel = GemmKernel::kTile;
    return c;
  }
  c.skinny = skinny_ok && !w_tiled ? skinny_plan(M, N, steps, cus, false) : skinny_t;
  // whole 256-row tiles; the last one does not write rows past M and reads no activation row past
  // a_rows (lanes that would are pointed at the last readable row)
  c.kernel = whole_tiles && (!skinny_ok || whole_us < c.skinny.us) ? GemmKernel::kWhole : GemmKernel::kSkinny;
  return c;
}

// The choice for the host alone: out[0] the kernel (MG_KERNEL_*), out[1] features and out[2] tokens per workgroup.
void mixed_gemm_choice(int M, int N, int KN, int KS, int KO, bool w_tiled, int cus, int out[3]) {
  const DecodeSeg d4 = {nullptr, nullptr, nullptr, nullptr, KN / 32, ceil_div(KN, 128)};
  const DecodeSeg d6 = {nullptr, nullptr, nullptr, nullptr, KS / 32, ceil_div(KS, 128)};
  const DecodeSeg d8 = {nullptr, nullptr, nullptr, nullptr, KO / 32, ceil_div(KO, 128)};
  const GemmChoice c = choose_gemm(d4, d6, d8, M, N, KN, KS, KO, w_tiled, cus);
  out[0] = (int)c.kernel;
  switch (c.kernel) {
    case GemmKernel::kDecode: out[1] = 16 * c.decode_f; out[2] = 16; break;
    case GemmKernel::kSkinny: out[1] = 16 * c.skinny.f; out[2] = 16 * c.skinny.g; break;
    case GemmKernel::kTile: out[1] = c.tile.tf; out[2] = c.tile.tt; break;
    case GemmKernel::kWhole: out[1] = out[2] = 256; break;
    default: out[1] = out[2] = 0;
  }
}

// a_rows: token rows for which the activation codes and scales are readable (>= M).  a_staged: the codes are stage by stage, of so many rows
// (see launch_reorder_quant); for whole and small tiles alone.
hipError_t launch_mixed_gemm(const uint8_t* an, const uint8_t* bn, const uint8_t* as_, const uint8_t* bs,
                             const uint8_t* ao, const uint8_t* bo, const uint8_t* sfan, const uint8_t* sfbn,
                             const uint8_t* sfas, const uint8_t* sfbs, const uint8_t* sfao, const uint8_t* sfbo, int M,
                             int a_rows, int a_staged, int N, int KN, int KS, int KO, unsigned flags, Epilogue ep, void* d,
                             hipStream_t stream) {
  if (M == 0 || N == 0) return hipSuccess;
  const bool w_tiled = (flags & 1u) != 0;   // MG_FLAG_W_TILED
  // tile-major weights exist only for shapes the 256x256 kernel takes
  if (w_tiled && (N % 256 != 0 || !mixed_gemm_256_supported(256, N, KN, KS, KO))) return hipErrorInvalidValue;
  const DecodeSeg d4 = {an, bn, sfan, sfbn, KN / 32, ceil_div(KN, 128)};
  const DecodeSeg d6 = {as_, bs, sfas, sfbs, KS / 32, ceil_div(KS, 128)};
  const DecodeSeg d8 = {ao, bo, sfao, sfbo, KO / 32, ceil_div(KO, 128)};
  DeviceLimits lim;
  if (hipError_t e = device_limits(&lim); e != hipSuccess) return e;
  const GemmChoice c = choose_gemm(d4, d6, d8, M, N, KN, KS, KO, w_tiled, lim.cus);
  if (a_staged != 0 && c.kernel != GemmKernel::kWhole && c.kernel != GemmKernel::kTile) return hipErrorInvalidValue;
  switch (c.kernel) {
    case GemmKernel::kDecode:
      return launch_decode(d4, d6, d8, M, N, w_tiled, c.decode_f, c.lds, ep, static_cast<uint16_t*>(d), stream);
    case GemmKernel::kSkinny:
      return launch_skinny(d4, d6, d8, M, N, w_tiled, c.skinny, ep, static_cast<uint16_t*>(d), stream);
    case GemmKernel::kTile:
      return launch_mixed_gemm_tile(an, bn, as_, bs, ao, bo, sfan, sfbn, sfas, sfbs, sfao, sfbo, M, a_rows, a_staged, N, KN, KS, KO, w_tiled,
                                    c.tile, ep, d, stream);
    case GemmKernel::kWhole:
      return launch_mixed_gemm_256(an, bn, as_, bs, ao, bo, sfan, sfbn, sfas, sfbs, sfao, sfbo, M, a_rows, a_staged, N, KN, KS, KO, w_tiled,
                                   ep, d, stream);
    default: return hipErrorInvalidValue;
  }
}

// Quantization and GEMM of a few tokens in one launch, where that is the faster way; *taken says whether it was.
// Every workgroup repeats the quantization, so it pays up to 16384 channels in all, up to 20480 for 5 tokens, 6 and 8 of them on row-major weights
// with two and four feature groups (120 shapes above 16384, two launches over one from HBM / from the caches: tile-major M = 3 ... 5 0.99 ... 1.13
// / 0.94 ... 1.08, 6 0.98 ... 1.07 / 0.95 ... 1.00, 7 0.98 ... 1.04 / 0.93 ... 0.97, 8 0.95 ... 1.05 / 0.92 ... 0.99; row-major with one group M = 4 and 5 1.02 ... 1.06 /
// 1.00 ... 1.03, 6 1.00 / 0.99, 8 0.96 / 0.93, with two M = 6 1.13 / 1.01, 7 1.09 / 0.97, with four M = 8 1.12 / 1.04), with RMSNorm up to 10240
// (M = 3, N = 4096 / 14336, K = 4096 9.0 against 9.0 / 12.2 against 11.4, but 10.5 against
// 11.1 with the weights in the caches, N = 13312), from 5 tokens on, where a token's norm is one wave's work, 8192 (M = 8, K = 1024 level, K =
// 2048 7.6 against 8.8), for rows of at most 8192 (M = 1, K = 14336, with longer rings: 13.7 against 14.0), and in one round of workgroups.
hipError_t launch_token_linear(const void* x, const int16_t* idx, const void* gamma, float eps, const uint8_t* bn, const uint8_t* bs,
                               const uint8_t* bo, const uint8_t* sfbn, const uint8_t* sfbs, const uint8_t* sfbo, int M, int N,
                               int KN, int KS, int KO, bool w_tiled, Epilogue ep, void* d, hipStream_t stream, bool* taken) {
  *taken = false;
  const int K = KN + KS + KO;
  // (row-major weight codes are addressed with 32-bit offsets; the copies of gamma want it aligned)
  const int widest = KN > KS ? (KN > KO ? KN : KO) : (KS > KO ? KS : KO);
  if (M < 1 || M > kTokenRows || K == 0 || K > 8192 || M * K > (gamma ? (M > 4 ? 8192 : 10240) : 20480) || N == 0 || (!w_tiled && (size_t)N * (size_t)(widest / 2) >= ((size_t)1 << 32)) ||
      (reinterpret_cast<uintptr_t>(gamma) & 15u))
    return hipSuccess;
  // tile-major weights exist only for shapes the 256x256 kernel takes
  if (w_tiled && (N % 256 != 0 || !mixed_gemm_256_supported(256, N, KN, KS, KO))) return hipErrorInvalidValue;
  DeviceLimits lim;
  if (hipError_t e = device_limits(&lim); e != hipSuccess) return e;
  const DecodeSeg d4 = {nullptr, bn, nullptr, sfbn, KN / 32, ceil_div(KN, 128)};
  const DecodeSeg d6 = {nullptr, bs, nullptr, sfbs, KS / 32, ceil_div(KS, 128)};
  const DecodeSeg d8 = {nullptr, bo, nullptr, sfbo, KO / 32, ceil_div(KO, 128)};
  const int total = d4.steps + d6.steps + d8.steps;
  const int f = ceil_div(N, 16) <= lim.cus ? 1 : (ceil_div(N, 32) <= lim.cus ? 2 : 4);
  const int grid = w_tiled ? ceil_div(N, 16 * f) : ceil_div(N, 128) * (8 / f);
  if (grid > lim.cus || (M * K > 16384 && M > (w_tiled ? 5 : 4 + f))) return hipSuccess;
  TokenLds L;
  int pos = 4 * 1024 * (f == 1 ? kTokenSlots<1> : (f == 2 ? 2 * kTokenSlots<2> : 4 * kTokenSlots<4>));
  auto take = [&](int bytes) { const int at = pos; pos += round_up_1k(bytes); return at; };
  L.x = take(M * K * 2); L.idx = take(K * 2); L.gamma = gamma ? take(K * 2) : 0;
  L.sw0 = take(d4.steps * f * 64); L.sw1 = take(d6.steps * f * 64); L.sw2 = take(d8.steps * f * 64);
  L.sx0 = take(d4.steps * 4 * kTokenRows); L.sx1 = take(d6.steps * 4 * kTokenRows); L.sx2 = take(d8.steps * 4 * kTokenRows);
  L.q0 = take(M * d4.nblk * 16); L.q1 = take(M * d6.nblk * 24); L.q2 = take(M * d8.nblk * 32);
  L.sums = take(128);   // also what a last, partial step reads past the last codes (and drops)
  L.total = pos;
  if (pos > lim.lds_bytes) return hipSuccess;
  auto launch = [&](auto f_c, auto wt_c, auto norm_c) {
    const auto kernel = mixed_gemm_token_kernel<decltype(f_c)::value, decltype(wt_c)::value, decltype(norm_c)::value>;
    if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lim.lds_bytes); e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * kTokenWaves), (size_t)L.total, stream, static_cast<const uint8_t*>(x),
                       static_cast<const uint8_t*>(gamma), reinterpret_cast<const uint8_t*>(idx), eps, K, d4, d6, d8, M, N,
                       (total + 3) / 4, L, ep, static_cast<uint16_t*>(d));
    return hipGetLastError();
  };
  auto with_norm = [&](auto f_c, auto wt_c) {
    return gamma ? launch(f_c, wt_c, std::true_type{}) : launch(f_c, wt_c, std::false_type{});
  };
  auto with_layout = [&](auto f_c) { return w_tiled ? with_norm(f_c, std::true_type{}) : with_norm(f_c, std::false_type{}); };
  *taken = true;
  if (f == 1) return with_layout(std::integral_constant<int, 1>{});
  if (f == 2) return with_layout(std::integral_constant<int, 2>{});
  return with_layout(std::integral_constant<int, 4>{});
}

}  // namespace mg
