// Reorder-quantize kernels for gfx950: gather bf16 channels by a reorder index,
// then per-32-element power-of-two (E8M0) scaling and quantization into packed
// MXFP4 (E2M1) / MXFP6 (E3M2) / MXFP8 (E4M3) segments.
//
// Semantics follow the reference kernels reorder_bf16_mixed_kernel
// (src/reorder.cu:94-269) and reorder_bf16_fp4_kernel (src/reorder.cu:271-432):
//   scale  = 2^e, e = min{e : amax <= MAX * 2^e}  (= ceil(log2(amax/MAX)), :180),
//            0.5 for an all-zero block (:179); E8M0 byte = e + 127
//   code   = RNE_fmt( bf16( clamp( roundf(x / scale) ) ) )   (:221-248)
// The design is not the reference's: rows go global -> LDS directly, as they are
// in memory, one or two lanes own a 32-element block and gather its channels
// from there, the scale exponent comes from integer arithmetic on the float
// bits, and the element conversion is done by the gfx950 cvt_scalef32
// instructions on the already integer-rounded values.
#include <type_traits>

#include "mg_common.h"
#include "quantize.h"

namespace mg {

namespace {

__device__ __forceinline__ unsigned perm(unsigned hi, unsigned lo, unsigned sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}

// Stores of the codes and the scale byte.  COUNTED: as inline assembly, one instruction each, so that a kernel
// which waits with s_waitcnt vmcnt(n) on older requests knows exactly how many stores it has issued since;
// the codes go out as streaming (nt) stores, which leave the L2 while the kernel runs instead of in the
// write-back at its end, the scale bytes as ordinary stores (the 32 rows that share a 128-byte line of a scale
// atom are written by different workgroups; the L2 merges them).  KEEP: ordinary stores for the codes too -- for
// the fused call, whose GEMM reads them next: the quantizer is then about a microsecond slower and the GEMM five
// to six faster (measured on M = 4096, K = 4096, N = 14336).
template <bool COUNTED, bool KEEP = false>
__device__ __forceinline__ void store16(uint8_t* q, v4u v) {
  if constexpr (COUNTED && KEEP) asm volatile("global_store_dwordx4 %0, %1, off" : : "v"(q), "v"(v) : "memory");
  else if constexpr (COUNTED) asm volatile("global_store_dwordx4 %0, %1, off nt" : : "v"(q), "v"(v) : "memory");
  else *reinterpret_cast<v4u*>(q) = v;
}
template <bool COUNTED, bool KEEP = false>
__device__ __forceinline__ void store8(uint8_t* q, v2u v) {
  if constexpr (COUNTED && KEEP) asm volatile("global_store_dwordx2 %0, %1, off" : : "v"(q), "v"(v) : "memory");
  else if constexpr (COUNTED) asm volatile("global_store_dwordx2 %0, %1, off nt" : : "v"(q), "v"(v) : "memory");
  else *reinterpret_cast<v2u*>(q) = v;
}
template <bool COUNTED>
__device__ __forceinline__ void store1(uint8_t* q, int byte) {
  if constexpr (COUNTED) asm volatile("global_store_byte %0, %1, off" : : "v"(q), "v"(byte) : "memory");
  else *q = (uint8_t)byte;
}
// store instructions a wave issues per row for a block format (plus one for the scale byte)
__device__ __forceinline__ constexpr int code_stores(int fmt) { return fmt == kFmtE2M1 ? 1 : (fmt == kFmtE3M2 ? 3 : 2); }

// Quantize one gathered block (32 floats holding bf16 values) and store its codes and scale.
// Everything up to the integer-valued v[] is the same instruction stream for the three
// formats (a wave that straddles a segment boundary runs it once, not once per format); only
// the final conversion and store differ.
template <bool COUNTED = false, bool KEEP = false>
__device__ __forceinline__ void quantize_store(const float (&f)[32], int fmt, uint8_t* __restrict__ q,
                                               uint8_t* __restrict__ sf) {
  float amax = 0.0f;
#pragma unroll
  for (int p = 0; p < 32; p += 2) amax = __builtin_fmaxf(__builtin_fmaxf(amax, __builtin_fabsf(f[p])), __builtin_fabsf(f[p + 1]));
  const int byte = scale_byte(amax, fmt);
  const float rs1 = __uint_as_float(((unsigned)(254 - byte) << 23) | 0x800u);   // 2^(127 - byte) * (1 + 2^-12)
  float v[32];
#pragma unroll
  for (int p = 0; p < 32; ++p) v[p] = round_scaled(f[p], rs1);
  store1<COUNTED>(sf, byte);

  if (fmt == kFmtE2M1) {
    v4u out;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned w = 0;
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 0], v[8 * j + 1], 1.0f, 0);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 2], v[8 * j + 3], 1.0f, 1);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 4], v[8 * j + 5], 1.0f, 2);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[8 * j + 6], v[8 * j + 7], 1.0f, 3);
      out[j] = w;
    }
    store16<COUNTED, KEEP>(q, out);
  } else {
    // the bf16 hop of the reference (src/reorder.cu:223) is a real rounding above 256
    v32bf h;
#pragma unroll
    for (int p = 0; p < 32; ++p) h[p] = (__bf16)v[p];
    if (fmt == kFmtE3M2) {
      // the ISA calls E3M2 "bf6" (its "fp6" is E2M3)
      const v6u w = __builtin_amdgcn_cvt_scalef32_pk32_bf6_bf16(h, 1.0f);
      store8<COUNTED, KEEP>(q, v2u{w[0], w[1]});
      store8<COUNTED, KEEP>(q + 8, v2u{w[2], w[3]});
      store8<COUNTED, KEEP>(q + 16, v2u{w[4], w[5]});
    } else {
      unsigned out[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const v2bf lo = {h[4 * j + 0], h[4 * j + 1]};
        const v2bf hi = {h[4 * j + 2], h[4 * j + 3]};
        v2s z = {0, 0};
        z = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(z, lo, 1.0f, false);
        z = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(z, hi, 1.0f, true);
        out[j] = __builtin_bit_cast(unsigned, z);
      }
      store16<COUNTED, KEEP>(q, v4u{out[0], out[1], out[2], out[3]});
      store16<COUNTED, KEEP>(q + 16, v4u{out[4], out[5], out[6], out[7]});
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The kernel (activations and weights): rows go global -> LDS directly.
//
// A workgroup owns rows first, first + gridDim.x, ... and a ring of NS row slots in LDS (row-major, as in
// memory).  The rows of the first NS iterations are requested before anything else happens
// (global_load_lds_dwordx4: no staging registers, nothing to wait for in the requesting wave); the slot a row
// leaves is refilled one iteration later, behind the barrier that also publishes the next row.  A lane gathers
// its channels with ds_read_u16_d16_hi, which puts the bf16 into the upper half of a register whose lower half
// is zero and stays zero -- the value is a float without a conversion instruction.
//
// EPL = 32: one lane per 32-element block (K/32 lanes).  EPL = 16: two lanes per block (K/16 lanes, K up to
// 16384): half the dependent work per lane and row, which is what bounds small problems -- the time from a
// row's arrival to its last store; the block's absmax is one cross-lane step.
//
// Everything a wave requests or stores goes through inline assembly, one instruction each, so that the waits
// on a row (s_waitcnt vmcnt(n): requests and stores complete in order) can count what was issued after it.
//
// T > 0: blockDim.x == T and the slot offsets are immediates of the LDS reads; T == 0: any blockDim.x, the
// slot offset is added to the addresses per row.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void dma16(const uint8_t* base, unsigned voff, unsigned lds_off) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               : : "v"(voff), "s"(base), "s"(lds_off) : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void wait_vm_imm() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

// s_waitcnt vmcnt(n) for a wave-uniform n: the wave's n most recent requests and stores may still be in flight
__device__ __forceinline__ void wait_vm(int n) {
  switch (n) {
#define MG_VM_CASE(N) case N: wait_vm_imm<N>(); break;
    MG_VM_CASE(0) MG_VM_CASE(1) MG_VM_CASE(2) MG_VM_CASE(3) MG_VM_CASE(4) MG_VM_CASE(5) MG_VM_CASE(6) MG_VM_CASE(7)
    MG_VM_CASE(8) MG_VM_CASE(9) MG_VM_CASE(10) MG_VM_CASE(11) MG_VM_CASE(12) MG_VM_CASE(13) MG_VM_CASE(14) MG_VM_CASE(15)
    MG_VM_CASE(16) MG_VM_CASE(17) MG_VM_CASE(18) MG_VM_CASE(19) MG_VM_CASE(20) MG_VM_CASE(21) MG_VM_CASE(22) MG_VM_CASE(23)
    MG_VM_CASE(24) MG_VM_CASE(25) MG_VM_CASE(26) MG_VM_CASE(27) MG_VM_CASE(28) MG_VM_CASE(29) MG_VM_CASE(30) MG_VM_CASE(31)
    MG_VM_CASE(32) MG_VM_CASE(33) MG_VM_CASE(34) MG_VM_CASE(35) MG_VM_CASE(36) MG_VM_CASE(37) MG_VM_CASE(38) MG_VM_CASE(39)
#undef MG_VM_CASE
    default: wait_vm_imm<40>(); break;   // n > 40: wait for a little more than necessary
  }
}

// 16 gathered channels: u[p] <- bf16 at LDS address ga[p] + OFF (an immediate), as the upper half.  OFF < 0 (the
// kernel with a run-time workgroup size, 1024 lanes and 128 registers each, which spills): at ga[p] + add, through
// reads the compiler sees and waits for itself, so that a spilled register is always a loaded one.
template <int OFF>
__device__ __forceinline__ void gather16(unsigned (&u)[16], const unsigned (&ga)[16], unsigned add) {
#pragma unroll
  for (int p = 0; p < 16; ++p) {
    if constexpr (OFF >= 0) {
      asm volatile("ds_read_u16_d16_hi %0, %1 offset:%2" : "+v"(u[p]) : "v"(ga[p]), "n"(OFF));
    } else {
      typedef __attribute__((address_space(3))) const uint16_t* lds_u16;
      u[p] = (unsigned)*reinterpret_cast<lds_u16>((size_t)(ga[p] + add)) << 16;
    }
  }
}
// the reads above are invisible to the compiler's own wait insertion: wait here, with the registers tied to the wait
__device__ __forceinline__ void gather_wait(unsigned (&u)[16]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]), "+v"(u[4]), "+v"(u[5]), "+v"(u[6]), "+v"(u[7]),
                 "+v"(u[8]), "+v"(u[9]), "+v"(u[10]), "+v"(u[11]), "+v"(u[12]), "+v"(u[13]), "+v"(u[14]), "+v"(u[15]));
}


// Codes and scale byte of half a block to memory, counted stores.
template <bool KEEP>
struct StoreHalf {
  uint8_t* q;    // of the block
  uint8_t* sf;
  int half;
  __device__ __forceinline__ void scale(int byte) const { store1<true>(sf, byte); }
  __device__ __forceinline__ void codes(v2u v) const { store8<true, KEEP>(q + half * 8, v); }
  __device__ __forceinline__ void codes(v3u v) const {
    if constexpr (KEEP) asm volatile("global_store_dwordx3 %0, %1, off" : : "v"(q + half * 12), "v"(v) : "memory");
    else asm volatile("global_store_dwordx3 %0, %1, off nt" : : "v"(q + half * 12), "v"(v) : "memory");
  }
  __device__ __forceinline__ void codes(v4u v) const { store16<true, KEEP>(q + half * 16, v); }
};

// Which rows a workgroup takes (see the kernel).  With a whole number `a` of rows per workgroup the plain schedule
// is `a` full iterations; the skewed one is a - 1 full iterations, one without the last generation of workgroups
// and one with the first generation only.  A CU's workgroups are dispatched one generation (gridDim.x / per-CU
// count) after the other and its memory requests are served in the order they were made, so the workgroup
// dispatched last gets its first row after everything its neighbours asked for at their start: it runs a row
// or two behind them for the whole launch, and the kernel ends when it does.  One row less for it and one more
// for the first generation evens that out (c1, 4 rows per workgroup: 10.2 -> 9.65 us).
struct RowSchedule {
  int head;       // iterations in which every workgroup takes a row
  int width[3];   // then: the first width[j] workgroups take one (0: nobody)
};

// TILED (weights): the codes go out in the tile-major order of mg_tile_weights, and rows past src_rows (up to whole
// tiles) are quantized as zeros.  A row's stores are then 64-byte pieces 16 KB apart instead of one run; the two rows that
// share a line go to workgroups of one XCD, whose L2 joins them, and the pass is as fast as the row-major one:
// W[14336, 4096] 38.7 us for quantizing and tiling one after the other, 24.6 in one pass (6.0 TB/s of what it has to move).
// STAGED: a_staged says whether the codes go stage by stage (see launch_reorder_quant), without a branch, and the addresses are worked out while the index
// is on its way.  Behind the wait for it, where the compiler does that by itself (with an instance for each order, too), M = 1055, N = 384, K = 4096 with RMSNorm
// is 14.35 us instead of 14.12, M = 1024, N = K = 4096 18.3 instead of 18.05.
template <int EPL, int T, int NS, bool IS_W, int MAXT, bool KEEP = false, bool NORM = false, bool TILED = false, bool STAGED = KEEP>
__global__ void __launch_bounds__(MAXT)
reorder_quant_dma_kernel(const uint8_t* __restrict__ x, const int16_t* __restrict__ idx, int rows, int K, int KN, int KS,
                         int KO, uint8_t* __restrict__ qn, uint8_t* __restrict__ qs, uint8_t* __restrict__ qo,
                         uint8_t* __restrict__ sfn, uint8_t* __restrict__ sfs, uint8_t* __restrict__ sfo, RowSchedule sched,
                         const uint16_t* __restrict__ gamma, float eps, double inv_k, int src_rows, int a_staged,
                         unsigned* __restrict__ verdict) {
  extern __shared__ __align__(16) uint8_t lds[];
  __shared__ double row_sums[NORM ? 2 : 1][NORM ? MAXT / 64 : 1];   // RMSNorm: the waves' sums of squares, by row parity
  static_assert(EPL == 32 || EPL == 16, "one or two lanes per block");
  constexpr int kPieces = EPL / 8;   // 16-byte pieces of a row (and of the index) per lane
  constexpr int kParts = EPL / 16;   // gathers of 16 per lane and row
  constexpr bool kImm = T > 0;
  // RMSNorm: two lanes per block normalize the channels they have gathered; one lane per block, whose gathered weights would take
  // 32 registers, normalizes the row in place before the gather
  constexpr bool kLate = NORM && EPL == 16;
  static_assert(!kLate || kImm, "the weight's loads are counted");
  static_assert(!kImm || (kLate ? NS : NS - 1) * 2 * EPL * T <= 65535, "slot offsets must fit the LDS instructions' immediate");
  const int tid = threadIdx.x;
  const int nthr = kImm ? T : (int)blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned stride = 2u * EPL * nthr;   // bytes per slot: kPieces copies of nthr x 16 bytes, at least one row
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int grid = gridDim.x;
  // Which row a workgroup starts with.  The scale bytes of 32 rows -- r % 32 in [8k, 8k + 8) for one k, any
  // (r / 32) % 4, of one group of 128 rows -- share a 128-byte line of a scale atom, and each row is written by
  // another workgroup.  Workgroups go to the 8 XCDs (one L2 each) round-robin by index, so the rows of a line
  // are given to workgroups of one XCD (row bits 3, 4, 7 = workgroup bits 0, 1, 2): its L2 then assembles the
  // whole line instead of eight L2s holding an eighth each until the write-back at the end of the kernel.
  int first = blockIdx.x;
  if (first < (grid & ~255)) {
    const int xcd = first & 7, y = (first >> 3) & 31;
    first = (first & ~255) | (y & 7) | ((xcd & 3) << 3) | (((y >> 3) & 3) << 5) | ((xcd >> 2) << 7);
  }
  // The rows of this workgroup: `sched.head` iterations in which every workgroup takes a row (iteration k: row
  // k * grid + first), then up to three iterations in which the first sched.width[j] workgroups do.
  const bool in_tail[3] = {first < sched.width[0], first < sched.width[1], first < sched.width[2]};
  const int count = sched.head + in_tail[0] + in_tail[1] + in_tail[2];
  auto row_of = [&](int k) {
    if (k < sched.head) return k * grid + first;
    int off = sched.head * grid, t = k - sched.head;   // the t-th tail iteration this workgroup is part of
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      if (in_tail[j]) {
        if (t == 0) break;
        --t;
      }
      off += sched.width[j];
    }
    return off + first;
  };
  const size_t row_bytes = (size_t)K * 2;
  // the row to read for a row of the result: past the last one that exists the last one again (its values are dropped)
  auto src_row = [&](int row) { return TILED ? min(row, src_rows - 1) : row; };

  // per-lane byte offsets of the lane's 16-byte pieces of a row (pieces past the row's end: the last one
  // again, into the slot's padding)
  const int nchunks = K >> 3;
  unsigned voff[kPieces];
#pragma unroll
  for (int it = 0; it < kPieces; ++it) voff[it] = (unsigned)min(it * nthr + tid, nchunks - 1) * 16u;
  const unsigned wave_lds = lds0 + (unsigned)wave * 1024u;
  auto request = [&](const uint8_t* base, unsigned slot_off) {
#pragma unroll
    for (int it = 0; it < kPieces; ++it) dma16(base, voff[it], wave_lds + slot_off + (unsigned)it * nthr * 16u);
  };

  // the lane's block and, with two lanes per block, its half
  const int b = EPL == 32 ? tid : tid >> 1;
  const int half = EPL == 32 ? 0 : tid & 1;
  const bool has_block = b < (K >> 5);

  // ---- everything this workgroup can have in flight, requested up front: the lane's EPL index entries (into
  //      registers), then the first NS rows
  v4u iv[kPieces];
  {
    const v4u* ip = reinterpret_cast<const v4u*>(idx + (size_t)(has_block ? b : 0) * 32 + half * 16);
    // (kernels with a compile-time workgroup size: as uncounted loads, waited for below; they compile without scratch
    // memory -- the build checks it --, so that no register is moved before its load has landed)
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
      if constexpr (kImm) asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(iv[q]) : "v"(ip + q) : "memory");
      else iv[q] = ip[q];
    }
  }
  // RMSNorm: the weights of this lane's pieces of a row (the same for every row).  kLate: uncounted loads, older than the rows
  // and there when the first one is; else ordinary loads, which the compiler waits for itself where they are first used (with
  // vmcnt(0): once, in the first row).
  v4u gv[kPieces];
  if constexpr (kLate) {
#pragma unroll
    for (int it = 0; it < kPieces; ++it)
      asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(gv[it]) : "v"(gamma + (size_t)min(it * nthr + tid, nchunks - 1) * 8) : "memory");
  }
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < count) request(x + (size_t)src_row(row_of(s)) * row_bytes, s * stride);
  if constexpr (NORM && !kLate) {
#pragma unroll
    for (int it = 0; it < kPieces; ++it)
      gv[it] = *reinterpret_cast<const v4u*>(gamma + (size_t)min(it * nthr + tid, nchunks - 1) * 8);
  }

  const int nbn = KN >> 5, nbs = KS >> 5;
  const int seg = b < nbn ? 0 : (b < nbn + nbs ? 1 : 2);
  const int j = seg == 0 ? b : (seg == 1 ? b - nbn : b - nbn - nbs);
  const int kseg = seg == 0 ? KN : (seg == 1 ? KS : KO);
  const int katoms = (kseg + 127) >> 7;
  const int fmt = IS_W ? kFmtE2M1 : (seg == 0 ? kFmtE2M1 : (seg == 1 ? kFmtE3M2 : kFmtE4M3));
  const int blk_bytes = fmt == kFmtE2M1 ? 16 : (fmt == kFmtE3M2 ? 24 : 32);
  size_t pitch = (size_t)(kseg >> 5) * blk_bytes;
  uint8_t* qbase = (seg == 0 ? qn : (seg == 1 ? qs : qo)) + j * blk_bytes;
  // Tile-major: a whole 128-wide step of a 256-row tile is 16 KB, of which row r has 64 bytes in copy block r % 16; the
  // blocks past the last whole step follow as `rows` rows of (blocks % 4).
  const int whole = kseg >> 7;
  const bool in_tile = TILED && (j >> 2) < whole;
  if constexpr (TILED) {
    qbase = (seg == 0 ? qn : (seg == 1 ? qs : qo)) + (in_tile ? (size_t)(j >> 2) * 16384 : (size_t)rows * whole * 64) + (j & 3) * 16;
    pitch = in_tile ? (size_t)whole * 16384 : (size_t)((kseg >> 5) & 3) * 16;   // per tile, or per row
  }
  uint8_t* sfbase = seg == 0 ? sfn : (seg == 1 ? sfs : sfo);
  // Stage by stage: of a_staged rows each.  Row by row (0) is the same with one row, but for the pitch: no branch.
  if constexpr (STAGED) {
    qbase = (seg == 0 ? qn : (seg == 1 ? qs : qo)) + (size_t)(j >> 2) * max(a_staged, 1) * (4 * blk_bytes) + (j & 3) * blk_bytes;
    pitch = (size_t)(a_staged == 0 ? kseg >> 5 : (j >> 2) < whole ? 4 : (kseg >> 5) & 3) * blk_bytes;
    asm volatile("" : "+v"(qbase), "+v"(pitch), "+v"(sfbase));   // before the wait for the index
  }

  // ---- the index entries are the oldest requests: they are there when at most the row copies are in flight
  wait_vm(kPieces * min(NS, count) + (kLate ? kPieces : 0));
  if constexpr (kPieces == 4) asm volatile("" : "+v"(iv[0]), "+v"(iv[1]), "+v"(iv[2]), "+v"(iv[3]));
  else asm volatile("" : "+v"(iv[0]), "+v"(iv[1]));
  // Is the index good?  A workgroup has all of it in its registers: the first one says so while its first rows arrive, every
  // wave for its part, in 16 words of host memory which the caller watches.  (A store that the counts of what is in flight leave
  // out makes their waits stricter, not laxer.)  N = 14336, K = 4096 with the entries copied to the host in front of the kernel,
  // 3.5 us and a gap on either side: 41.1 us, now 29.5.
  if constexpr (IS_W) {
    if (verdict != nullptr && blockIdx.x == 0) {
      bool bad = false;
#pragma unroll
      for (int q = 0; q < kPieces; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) bad |= (iv[q][e] & 0xffffu) >= (unsigned)K || (iv[q][e] >> 16) >= (unsigned)K;
      const unsigned word = __builtin_amdgcn_ballot_w64(bad) != 0 ? 2u : 1u;
      const int lane = tid & 63;
      if (lane < 16 && lane % (nthr >> 6) == wave) __hip_atomic_store(verdict + lane, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  // LDS byte addresses of the lane's gathered channels in slot 0.  An entry outside [0, K) is read as
  // channel K - 1, so that the gather stays inside the row whatever the index holds.
  unsigned ga[kParts][16];
#pragma unroll
  for (int q = 0; q < kPieces; ++q)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      ga[q >> 1][(q & 1) * 8 + e] =
          lds0 + min((e & 1) ? (iv[q][e >> 1] >> 16) : (iv[q][e >> 1] & 0xffffu), (unsigned)(K - 1)) * 2u;
  unsigned u[kParts][16];
#pragma unroll
  for (int h = 0; h < kParts; ++h)
#pragma unroll
    for (int p = 0; p < 16; ++p) u[h][p] = 0u;
  // store instructions this wave issues per row: the scale byte, and the codes once per format its lanes have
  const int fmt_or_none = has_block ? fmt : -1;
  const int row_stores =
      1 + (__builtin_amdgcn_ballot_w64(fmt_or_none == kFmtE2M1) ? (EPL == 32 ? code_stores(kFmtE2M1) : 1) : 0) +
      (__builtin_amdgcn_ballot_w64(fmt_or_none == kFmtE3M2) ? (EPL == 32 ? code_stores(kFmtE3M2) : 1) : 0) +
      (__builtin_amdgcn_ballot_w64(fmt_or_none == kFmtE4M3) ? (EPL == 32 ? code_stores(kFmtE4M3) : 1) : 0);

  unsigned gw[kLate ? 16 : 1];   // kLate: the weights of the lane's gathered channels, in the upper halves

  int i = 0;
  auto body = [&](auto slot_c) {
    constexpr int S = decltype(slot_c)::value;
    const int row = row_of(i);
    // Row i has landed when at most what was issued after its request is in flight (requests and stores complete
    // in order): the requests of the rows after it -- NS - 1 of them at the start, NS - 2 once refills follow the
    // iterations -- and the stores of the iterations since, at most NS - 1 of them.
    wait_vm(kPieces * min(i == 0 ? NS - 1 : NS - 2, count - 1 - i) + row_stores * min(i, NS - 1));
    if constexpr (NORM) {
      // RMSNorm of the row (the arithmetic of the usual fp32 implementation):
      //   var = fl32( (sum over the row of x^2, accumulated in fp64) / K )
      //   r   = fl32( 1 / sqrt( fl32(var + eps) ) )      (quotient and root to a unit in the last place of a double: rms_scale)
      //   y   = bf16( gamma * bf16( x * r ) )            (both products in fp32)
      // The fp64 sum makes the result independent of the order in which the lanes add their parts (up to the last
      // bit of a double, which the rounding to fp32 all but never sees).  A lane sums over the pieces it copied.
      // kLate: one barrier per row as without RMSNorm, nothing written back, and the vector ALUs, which bound it, have 220
      // instructions per row and wave next to the quantizer's 110 instead of 280: M = 4096, K = 4096 17.1 us normalized in place, now
      // 15.8; 8192 rows 28.9 -> 26.5, 1024 7.1 -> 6.7.
      uint8_t* slot = lds + S * stride;
      v4u a[kPieces];
      double part[4] = {0.0, 0.0, 0.0, 0.0};   // four chains: one chain of dependent fp64 fmas would wait for each in turn
#pragma unroll
      for (int it = 0; it < kPieces; ++it) {
        a[it] = *reinterpret_cast<const v4u*>(slot + (size_t)(it * nthr + tid) * 16);
        if (it * nthr + tid < nchunks) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const unsigned d = a[it][e];
            const double lo = (double)__uint_as_float(d << 16), hi = (double)__uint_as_float(d & 0xffff0000u);
            part[e] = __builtin_fma(lo, lo, part[e]);
            part[e] = __builtin_fma(hi, hi, part[e]);
          }
        }
      }
      double ss = wave_sum((part[0] + part[1]) + (part[2] + part[3]));
      if ((tid & 63) == 0) row_sums[i & 1][tid >> 6] = ss;
      if constexpr (kLate) {
        if (i == 0) {   // the weights to LDS, behind the row slots, for the other lanes
#pragma unroll
          for (int it = 0; it < kPieces; ++it) {
            asm volatile("" : "+v"(gv[it]));   // (older than the row: landed)
            *reinterpret_cast<v4u*>(lds + NS * stride + (size_t)(it * nthr + tid) * 16) = gv[it];
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the sum is in the LDS (a raw barrier implies no wait of the compiler's)
      asm volatile("s_barrier" ::: "memory");   // also: every wave's copies of row i have landed, every wave is past its gather of row i - 1
      if (i >= 1 && i - 1 + NS < count)
        request(x + (size_t)src_row(row_of(i + NS - 1)) * row_bytes, ((S + NS - 1) % NS) * stride);
      if constexpr (!kLate) {
        double tot = 0.0;
        for (int w = 0; w < (nthr >> 6); ++w) tot += row_sums[i & 1][w];
        const float rn = rms_scale(tot, K, inv_k, eps);
#pragma unroll
        for (int it = 0; it < kPieces; ++it) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            a[it][e] = rms_apply(a[it][e], gv[it][e], rn);
          }
          if (it * nthr + tid < nchunks) *reinterpret_cast<v4u*>(slot + (size_t)(it * nthr + tid) * 16) = a[it];
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("s_barrier" ::: "memory");   // the normalized row is complete
      }
    } else {
      asm volatile("s_barrier" ::: "memory");
      // every wave is past its gather of row i - 1: refill that row's slot
      if (i >= 1 && i - 1 + NS < count)
        request(x + (size_t)src_row(row_of(i + NS - 1)) * row_bytes, ((S + NS - 1) % NS) * stride);
    }
    // (the sums of row i: written again, for row i + 2, behind the barrier of row i + 1)
    float rn = 0.0f;
    if constexpr (kLate) {
      double tot = 0.0;
      for (int w = 0; w < (nthr >> 6); ++w) tot += row_sums[i & 1][w];
      rn = rms_scale(tot, K, inv_k, eps);
      if (i == 0) {
        if (has_block) gather16<NS * 2 * EPL * T>(u[0], ga[0], 0u);
        gather_wait(u[0]);
#pragma unroll
        for (int p = 0; p < 16; ++p) {
          gw[p] = u[0][p];
          u[0][p] = 0u;
        }
      }
    }
    if (has_block) {
      constexpr int kOff = kImm ? S * 2 * EPL * T : -1;
#pragma unroll
      for (int h = 0; h < kParts; ++h) gather16<kOff>(u[h], ga[h], S * stride);
#pragma unroll
      for (int h = 0; h < kParts; ++h) gather_wait(u[h]);
      uint8_t* q = qbase + (size_t)row * pitch;
      if constexpr (TILED) {
        if (in_tile) {
          const int h = (row >> 4) & 15;   // rows 16 h ... of the tile: lane quad h / 2 + 8 (h % 2) of the copy block
          q = qbase + (size_t)(row >> 8) * pitch + (row & 15) * 1024 + ((h >> 1) + 8 * (h & 1)) * 64;
        }
        if (row >= src_rows) {   // workgroup-uniform
#pragma unroll
          for (int h = 0; h < kParts; ++h)
#pragma unroll
            for (int p = 0; p < 16; ++p) u[h][p] = 0u;
        }
      }
      uint8_t* sf = sfbase + sf_offset(row, j, katoms);
      if constexpr (EPL == 32) {
        float f[32];
#pragma unroll
        for (int p = 0; p < 32; ++p) f[p] = __uint_as_float(u[p >> 4][p & 15]);
        quantize_store<true, KEEP>(f, fmt, q, sf);
      } else {
        float f[16];
#pragma unroll
        for (int p = 0; p < 16; ++p) f[p] = __uint_as_float(u[0][p]);
        if constexpr (kLate)
#pragma unroll
          for (int p = 0; p < 16; p += 2) rms_apply(f[p], f[p + 1], gw[p], gw[p + 1], rn);
        quantize_half(f, fmt, half, StoreHalf<KEEP>{q, sf, half});
      }
    }
  };
  auto run = [&](auto self, auto slot_c) -> void {
    constexpr int S = decltype(slot_c)::value;
    body(slot_c);
    ++i;
    if constexpr (S + 1 < NS) {
      if (i < count) self(self, std::integral_constant<int, S + 1>{});
    }
  };
  while (i < count) run(run, std::integral_constant<int, 0>{});
}

// ---------------------------------------------------------------------------------------------
// Few rows: a workgroup quantizes 16 T channels of one row (two lanes per block) and nothing else.  A call of few rows is the latency of
// one: launch, index and row on their way, gather, arithmetic, stores.  Here a long row's last three are spread over several CUs -- each
// copies the whole row, since the gathered channels may lie anywhere in it, but only its part of the index --, and a short one is spared
// the schedule and the ring of rows.  The launch grid is 8 x parts x rows / 8: workgroups go to the 8 XCDs round-robin, so the parts
// of a row share an L2, which fetches it once (dealt out one by one, 128 rows of 14336 took 5.1 us instead of 3.5, of 28672 10.1 instead of 5.9).
// us, rows in the caches, the kernel above -> T = 256:
//   rows 16: K = 1024 2.65 -> 2.50, 4096 3.04 -> 2.82, 8192 3.25 -> 2.76, 14336 4.08 -> 2.96, 18944 4.79 -> 3.11, 28672 5.39 -> 3.17
//   rows 128: K = 1024 2.69 -> 2.54, 4096 3.19 -> 2.98, 8192 3.33 -> 2.87, 14336 4.38 -> 3.48, 18944 5.07 -> 4.10
// Layer calls, us: M = 32, N = 4096, K = 14336 13.6 -> 12.3; M = 100, N = K = 8192 16.6 -> 14.7 (some of it the GEMM's).
// With RMSNorm: rows 16: K = 2048 3.54 -> 3.35, 5120 4.30 -> 3.80, 8192 4.50 -> 4.01, 14336 5.78 -> 4.45.  (Gathering in front of the
// sum, with a barrier more, is level.)
// ---------------------------------------------------------------------------------------------
// STAGED: the codes stage by stage (see launch_reorder_quant; as an argument 0.2 us of every other call).
template <int T, bool KEEP, bool NORM, bool STAGED>
__global__ void __launch_bounds__(T)
reorder_quant_part_kernel(const uint8_t* __restrict__ x, const int16_t* __restrict__ idx, int rows, int K, int KN, int KS, int KO,
                          uint8_t* __restrict__ qn, uint8_t* __restrict__ qs, uint8_t* __restrict__ qo, uint8_t* __restrict__ sfn,
                          uint8_t* __restrict__ sfs, uint8_t* __restrict__ sfo, const uint8_t* __restrict__ gamma, float eps, double inv_k, int a_staged) {
  extern __shared__ __align__(16) uint8_t lds[];
  __shared__ double row_sums[NORM ? T / 64 : 1];   // RMSNorm: the waves' sums of squares
  const int tid = threadIdx.x, row = (int)blockIdx.z * 8 + (int)blockIdx.x;
  if (row >= rows) return;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int b = (int)blockIdx.y * (T / 2) + (tid >> 1), half = tid & 1;
  const bool has_block = b < (K >> 5);
  v4u iv[2];
  const v4u* ip = reinterpret_cast<const v4u*>(idx + (size_t)(has_block ? b : 0) * 32 + half * 16);
  asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(iv[0]) : "v"(ip) : "memory");
  asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(iv[1]) : "v"(ip + 1) : "memory");
  const uint8_t* base = x + (size_t)row * K * 2;
  const int nchunks = K >> 3, copies = (nchunks + T - 1) / T;
  for (int it = 0; it < copies; ++it)   // (past the row's end: its last piece again, into the padding)
    dma16(base, (unsigned)min(it * T + tid, nchunks - 1) * 16u, lds0 + (unsigned)(it * T * 16 + wave * 1024));
  const unsigned weights = (unsigned)copies * T * 16;   // RMSNorm: its weight, behind the row
  if constexpr (NORM)
    for (int it = 0; it < copies; ++it)
      dma16(gamma, (unsigned)min(it * T + tid, nchunks - 1) * 16u, lds0 + weights + (unsigned)(it * T * 16 + wave * 1024));

  const int nbn = KN >> 5, nbs = KS >> 5;
  const int seg = b < nbn ? 0 : (b < nbn + nbs ? 1 : 2);
  const int j = seg == 0 ? b : (seg == 1 ? b - nbn : b - nbn - nbs);
  const int kseg = seg == 0 ? KN : (seg == 1 ? KS : KO);
  const int fmt = seg == 0 ? kFmtE2M1 : (seg == 1 ? kFmtE3M2 : kFmtE4M3);
  const int blk_bytes = fmt == kFmtE2M1 ? 16 : (fmt == kFmtE3M2 ? 24 : 32);
  uint8_t* q = (seg == 0 ? qn : (seg == 1 ? qs : qo)) + (size_t)row * ((kseg >> 5) * blk_bytes) + j * blk_bytes;
  if constexpr (STAGED) {
    const int whole = kseg >> 7;
    const bool in_stage = (j >> 2) < whole;
    q = (seg == 0 ? qn : (seg == 1 ? qs : qo)) + (size_t)(in_stage ? j >> 2 : whole) * a_staged * (4 * blk_bytes) +
        (size_t)row * ((in_stage ? 4 : (kseg >> 5) & 3) * blk_bytes) + (j & 3) * blk_bytes;
  }
  uint8_t* sf = (seg == 0 ? sfn : (seg == 1 ? sfs : sfo)) + sf_offset(row, j, (kseg + 127) >> 7);
  wait_vm(copies * (NORM ? 2 : 1));   // the index
  asm volatile("" : "+v"(iv[0]), "+v"(iv[1]));
  unsigned ga[16], u[16];
#pragma unroll
  for (int p = 0; p < 16; ++p) {
    const unsigned pair = iv[p >> 3][(p & 7) >> 1];
    ga[p] = lds0 + min((p & 1) ? pair >> 16 : pair & 0xffffu, (unsigned)(K - 1)) * 2u;   // an entry outside [0, K): channel K - 1
    u[p] = 0u;
  }
  if constexpr (NORM) {   // every workgroup of a row sums all of it, a lane what it copied
    wait_vm(copies);
    double part[4] = {0.0, 0.0, 0.0, 0.0};
    for (int it = 0; it < copies; ++it) {
      const v4u a = *reinterpret_cast<const v4u*>(lds + (size_t)(it * T + tid) * 16);
      if (it * T + tid < nchunks) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double lo = (double)__uint_as_float(a[e] << 16), hi = (double)__uint_as_float(a[e] & 0xffff0000u);
          part[e] = __builtin_fma(lo, lo, part[e]);
          part[e] = __builtin_fma(hi, hi, part[e]);
        }
      }
    }
    const double sum = wave_sum((part[0] + part[1]) + (part[2] + part[3]));
    if ((tid & 63) == 0) row_sums[tid >> 6] = sum;
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the sum is in the LDS
  }
  wait_vm_imm<0>();
  asm volatile("s_barrier" ::: "memory");
  if (has_block) {
    gather16<0>(u, ga, 0u);
    [[maybe_unused]] unsigned gw[NORM ? 16 : 1];
    [[maybe_unused]] float rn = 0.0f;
    if constexpr (NORM) {
#pragma unroll
      for (int p = 0; p < 16; ++p) {
        ga[p] += weights;
        gw[p] = 0u;
      }
      gather16<0>(gw, ga, 0u);
      double tot = 0.0;
#pragma unroll
      for (int w = 0; w < T / 64; ++w) tot += row_sums[w];
      rn = rms_scale(tot, K, inv_k, eps);
      gather_wait(gw);
    }
    gather_wait(u);
    float f[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) f[p] = __uint_as_float(u[p]);
    if constexpr (NORM)
#pragma unroll
      for (int p = 0; p < 16; p += 2) rms_apply(f[p], f[p + 1], gw[p], gw[p + 1], rn);
    quantize_half(f, fmt, half, StoreHalf<KEEP>{q, sf, half});
  }
}

}  // namespace

// a_staged != 0 (activations whose codes are kept): the codes of a segment stage by stage, as a GEMM on tiles copies them -- per whole
// 128-wide stage `a_staged` rows (at least `rows`) of 64, 96 or 128 bytes one after the other, behind them rows of the blocks past the last whole
// stage.  A copy of 16 rows is then one run of whole lines; row-major, a row's 64 bytes of a stage are half a line and its 96 bytes lie in
// two, so that the GEMM fetched every line of E2M1 codes twice.  A row's stores are 64-byte pieces apart here; of neighbouring rows that share
// a line, the kernel for many rows has runs of eight on one XCD, whose L2 puts the lines together, the one for few rows each on another XCD, as parts of lines.  Layer calls, us, row-major -> stage by stage, one layer over and over / six in turn: M = 777, N = 5000, K = 5120 all
// E2M1 30.2 -> 28.4 / 30.2 -> 28.2; M = 2048, N = 4096, K = 14336 level (0.99 ... 1.014 times as fast over four machines) / 85.2 -> 79.8, row-major weights 88.7 -> 82.9 / 103 -> 95; M = 4096, N =
// 14336, K = 4096 126.2 -> 123.7 / 131.0 -> 126.7; M = 4096, N = K = 5120 74.9 -> 70.8 / 78.7 -> 73.0.  On small tiles (tile-major weights; before, long
// launches copied batches of rows): M = 256, N = K = 4096 10.9 -> 10.5 / 11.4 -> 11.0, M = 1024 19.6 -> 19.0 / 19.8 -> 19.4; M = 700, N = 4096, K = 5120 21.1
// -> 19.6 / 21.2 -> 19.5; M = 140, N = 18944, K = 8192 32.2 -> 30.7 / 44.5 -> 42.8.  The same bits in all of them.
// gamma != nullptr: RMSNorm with that weight and eps before the gather (activations only).  src_rows != 0 (weights only):
// codes in tile-major order, x has src_rows rows and the result `rows`, a multiple of 256.  verdict (weights only): 16 words, see the kernel.
template <bool IS_W>
hipError_t launch_reorder_quant(const void* x, const int16_t* idx, int rows, int K, int KN, int KS, int KO, uint8_t* qn,
                                uint8_t* qs, uint8_t* qo, uint8_t* sfn, uint8_t* sfs, uint8_t* sfo,
                                const void* gamma, float eps, bool keep_codes, int a_staged, int src_rows, unsigned* verdict, hipStream_t stream) {
  if (rows == 0 || K == 0) return hipSuccess;
  if ((gamma != nullptr && IS_W) || (verdict != nullptr && !IS_W) || (src_rows != 0 && (!IS_W || src_rows > rows || rows % 256 != 0))) return hipErrorInvalidValue;
  if (a_staged != 0 && (IS_W || !keep_codes || a_staged < rows)) return hipErrorInvalidValue;
  const uint16_t* gm = static_cast<const uint16_t*>(gamma);
  const int threads = ((K >> 5) + 63) & ~63;
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  DeviceLimits lim;
  if (hipError_t e = device_limits(&lim); e != hipSuccess) return e;
  hipError_t err = hipSuccess;
  // rows global -> LDS directly; NS row slots per workgroup, as many workgroups per CU as fit
  const int usable = lim.lds_bytes - 1024;   // the kernels' static LDS (row sums of the RMSNorm) stays below 1 KB
  auto launch_dma = [&](auto kernel, int epl, int NS, int nthreads, int max_per_cu, int most_waves = 16) {
    const int lds = (NS + (gm && epl == 16 ? 1 : 0)) * 2 * epl * nthreads;   // NS row slots, and the RMSNorm's weight
    if (lds > usable) { err = hipErrorInvalidValue; return; }
    int per_cu = usable / lds;
    per_cu = per_cu > max_per_cu ? max_per_cu : per_cu;
    const int by_waves = most_waves / (nthreads / 64);
    per_cu = per_cu > by_waves ? (by_waves < 1 ? 1 : by_waves) : per_cu;
    const int resident = lim.cus * per_cu;
    const int grid = rows < resident ? rows : resident;
    const int a = rows / grid, rem = rows - a * grid;
    RowSchedule sched;
    if (a >= 2 && per_cu >= 3 && grid == resident) {
      sched = RowSchedule{a - 1, {grid - lim.cus, lim.cus, rem}};
    } else {
      sched = RowSchedule{a - 1, {grid, rem, 0}};
    }
    err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), usable);
    if (err != hipSuccess) return;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(nthreads), (size_t)lds, stream, xb, idx, rows, K, KN, KS, KO, qn, qs, qo, sfn,
                       sfs, sfo, sched, gm, eps, 1.0 / K, src_rows, a_staged, verdict);
    err = hipGetLastError();
  };
  // Measured on M = 4096 ... 16384 rows of K = 3584 ... 18944: two row slots per workgroup, and per CU up to four
  // workgroups but no more than 16 waves (K = 5120: 3 x 5 waves, K = 12288: 2 x 6); more of either puts more requests
  // in front of a workgroup's first row and was slower.
  constexpr int kNS = 2;
  constexpr int kPerCu = 4;
  // Activations of 8192 < K <= 16384 with two lanes per block as well, i.e. 9 ... 16 waves per workgroup, where that is the faster way or level with the
  // rows in the caches, where the kernel before left them, and from HBM (us, one lane per block against two, from the caches / from HBM; two runs of one
  // side differ by 1 %).  Without RMSNorm:
  //   9 and 10 waves, one workgroup per CU: K = 9216 rows 256 4.4 against 4.4 / 4.4 against 4.45, 512 5.05, 5.4 / 6.1, 6.35, 640 7.2, 6.75 / 7.9, 7.55, 1024 8.2, 7.8 / 10.4, 8.9, 1025 8.2, 8.55 / 10.4, 9.4, 1600 9.9, 11.4 / 12.4, 12.25, 4096 22.2, 22.7 /
  //     24.6, 23.25; K = 10240 1024 8.1, 8.1 / 10.9, 9.3, 2048 13.1, 13.9 / 15.0, 14.4 (three per CU: 2048 rows of 9216 15 % slower than one lane);
  //   11 and 12 waves, two per CU: K = 12288 rows 256 4.55, 4.35 / 4.85, 4.65, 512 5.3, 5.6 / 6.9, 6.4, 1024 7.8, 7.6 / 10.0, 9.15, 1600
  //     11.0, 11.5 / 13.15, 12.4, 2048 13.7, 12.9 / 15.2, 14.2, 8192 45.9, 40.0 / 52.3, 49.1; K = 11008 1700 10.45, 10.7 / 12.55, 12.1, 4096 22.6, 20.8 / 25.4, 23.9;
  //   13 ... 16 waves, one per CU: K = 14336 rows 256 4.75, 4.75 / 5.2, 5.1, 320 5.5, 6.1 / 7.1, 6.95, 1024 9.1, 9.3 / 11.4, 11.3, 1600 12.8, 14.9 /
  //     15.3, 15.6, 3500 24.3, 24.6 / 27.7, 26.4, 4096 27.1, 27.2 / 32.0, 29.8, 8192 52.0, 49.5 / 61.3, 55.3; K = 12800 4096 25.3, 26.0 / 28.85, 27.15, 6144 36.4, 36.1 / 42.55,
  //     38.2; K = 15360 2560 20.1, 19.6 / 23.4, 22.2, K = 16384 2048 17.0, 17.35 / 20.2, 19.3, 3072 24.2, 22.9 / 27.6, 26.0 (two per CU: up to 15 % slower).
  // With RMSNorm, whose form for one lane per block normalizes the row in place: K = 9216 rows 512 9.8, 8.4 / 11.0, 8.8, 2048 28.5, 23.55 / 29.6,
  // 23.8; K = 12288 2048 30.4, 24.4 / 31.3, 24.7; K = 14336 128 6.35, 6.6 / 6.85, 6.65, 256 6.6, 6.85 / 7.3, 7.05, 257 10.3, 9.35 / 11.7, 9.5, 2048
  // 31.9, 28.4 / 33.0, 28.7; K = 12800 4096 51.0, 50.8 / 52.1, 51.0, 8192 93.8, 96.5 / 94.6, 96.6 (up to K = 15360: the LDS offsets of its three rows are
  // immediates).
  // Codes kept for the GEMM that follows, gain of two lanes per layer call (N = 4096): 9 and 10 waves, 512 rows -2 % / -1 %, 2048 and 4096 -1 % / 0.5 %; 11 and 12, up
  // to 900 rows 0 ... 4 % / 0 ... 4 %, from 1300 on 0 / 1 %; 13 ... 16, 256 rows 0 ... 2 % / 0 ... 2 %, 512 -1 % / 0, 2048 and 4096 -2 % / -1 ... 1 %.
  auto two_lanes = [&](int t2, bool norm, bool kept) {
    const int64_t r = rows, cus = lim.cus;
    if (norm) return t2 <= 768 || (t2 <= 960 && r > cus && (t2 > 832 || r <= 16 * cus));
    if (t2 > 1024) return false;
    // (no RMSNorm: fewer rows than CUs have gone to few_rows)
    if (t2 < 704) return !kept && 2 * r >= 5 * cus && r <= 4 * cus;
    if (t2 <= 768) return kept || r == cus || r >= 4 * cus;
    return r == cus || (!kept && r >= (t2 == 832 ? 24 : t2 == 896 ? 16 : 12) * cus);
  };
  // Fewer rows than CUs go to the kernel for few rows (from there on the workgroups of the other one are arranged so that an L2 puts the lines
  // of scales together: K = 4096, 256 rows 3.01 us there, 3.06 here, 255 rows 3.32 and 3.10); of more than 20480 channels three quarters as many (K =
  // 28672, 192 rows 6.60, 6.35, 255 7.16, 7.43).  Above 16384 channels and a workgroup of 4096 channels per CU with 8192 channels in each (K = 18944,
  // 64 rows 3.66 with 4096, 3.55, 255 5.85, 5.18 (the other kernel 5.93); K = 28672, 64 rows 3.89, 3.62, 128 5.88, 4.70 (5.92)).  With RMSNorm, where
  // every workgroup of a row sums all of it, at most a workgroup per CU (K = 8192, 128 rows 4.61, 4.14, 255 4.73, 4.98; K = 18944, 64 rows
  // 6.92, 8.49), and not 2048 < K <= 4096, on one measurement (alone 3.72, 3.67, but the layer call M = 8, N = 14336, K = 4096 10.7 -> 10.9 launched one by one; other
  // sizes of that band were not timed).
  const int64_t parts_of_4096 = (int64_t)rows * ((K + 4095) >> 12);
  auto few_rows = [&](bool norm) {
    // (the copies of the norm's weight want it aligned)
    if (norm) return (K <= 2048 || K > 4096) && parts_of_4096 <= lim.cus && (reinterpret_cast<uintptr_t>(gamma) & 15u) == 0;
    return K > 20480 ? (int64_t)rows * 4 <= (int64_t)lim.cus * 3 : rows < lim.cus;
  };
  // keep: the codes stay in the L2 for the kernel that reads them next (activations only); norm: RMSNorm of the row
  // before the gather (activations only; its codes are always kept: what follows a norm is the layer's GEMM)
  auto dispatch = [&](auto keep_c, auto norm_c, auto tiled_c) {
    constexpr bool TI = decltype(tiled_c)::value;
    constexpr bool KP = decltype(keep_c)::value;
    constexpr bool NM = decltype(norm_c)::value;
    const int t2 = ((K >> 4) + 63) & ~63;   // two lanes per block: K/16 lanes, rounded up to whole waves
    if constexpr (!IS_W) {
      auto parts = [&](auto t_c) {
        constexpr int T = decltype(t_c)::value;
        auto kernel = reorder_quant_part_kernel<T, KP, NM, false>;
        if constexpr (KP) {
          if (a_staged != 0) kernel = reorder_quant_part_kernel<T, KP, NM, true>;
        }
        const int lds = ((K >> 3) + T - 1) / T * T * 16 * (NM ? 2 : 1);   // the row, and the RMSNorm's weight
        if (lds > usable) { err = hipErrorInvalidValue; return; }
        err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), usable);
        if (err != hipSuccess) return;
        hipLaunchKernelGGL(kernel, dim3(8, ((K >> 4) + T - 1) / T, (rows + 7) / 8), dim3(T), (size_t)lds, stream, xb, idx, rows, K, KN, KS, KO, qn, qs, qo,
                           sfn, sfs, sfo, reinterpret_cast<const uint8_t*>(gm), eps, 1.0 / K, a_staged);
        err = hipGetLastError();
      };
      if (few_rows(NM)) {
        if constexpr (!NM) {
          if (K > 16384 && parts_of_4096 > lim.cus) return parts(std::integral_constant<int, 512>{});
        }
        return parts(std::integral_constant<int, 256>{});
      }
    }
    if (K <= 8192) {
      switch (t2) {
        case 64: launch_dma(reorder_quant_dma_kernel<16, 64, kNS, IS_W, 64, KP, NM, TI>, 16, kNS, 64, kPerCu); break;
        case 128: launch_dma(reorder_quant_dma_kernel<16, 128, kNS, IS_W, 128, KP, NM, TI>, 16, kNS, 128, kPerCu); break;
        case 192: launch_dma(reorder_quant_dma_kernel<16, 192, kNS, IS_W, 192, KP, NM, TI>, 16, kNS, 192, kPerCu); break;
        case 256: launch_dma(reorder_quant_dma_kernel<16, 256, kNS, IS_W, 256, KP, NM, TI>, 16, kNS, 256, kPerCu); break;
        case 320: launch_dma(reorder_quant_dma_kernel<16, 320, kNS, IS_W, 320, KP, NM, TI>, 16, kNS, 320, kPerCu); break;
        case 384: launch_dma(reorder_quant_dma_kernel<16, 384, kNS, IS_W, 384, KP, NM, TI>, 16, kNS, 384, kPerCu); break;
        case 448: launch_dma(reorder_quant_dma_kernel<16, 448, kNS, IS_W, 448, KP, NM, TI>, 16, kNS, 448, kPerCu); break;
        default: launch_dma(reorder_quant_dma_kernel<16, 512, kNS, IS_W, 512, KP, NM, TI>, 16, kNS, 512, kPerCu); break;
      }
    } else if (!IS_W && two_lanes(t2, NM, KP)) {
      if constexpr (!IS_W) {
        auto wide = [&](auto t_c) {
          constexpr int T2 = decltype(t_c)::value;
          if constexpr (NM ? T2 <= 960 : !KP || T2 >= 704)   // what two_lanes sends here
            launch_dma(reorder_quant_dma_kernel<16, T2, kNS, IS_W, T2, KP, NM, TI>, 16, kNS, T2, kPerCu, !NM && (T2 == 704 || T2 == 768) ? 24 : 16);
          else
            err = hipErrorInvalidValue;
        };
        switch (t2) {
          case 576: wide(std::integral_constant<int, 576>{}); break;
          case 640: wide(std::integral_constant<int, 640>{}); break;
          case 704: wide(std::integral_constant<int, 704>{}); break;
          case 768: wide(std::integral_constant<int, 768>{}); break;
          case 832: wide(std::integral_constant<int, 832>{}); break;
          case 896: wide(std::integral_constant<int, 896>{}); break;
          case 960: wide(std::integral_constant<int, 960>{}); break;
          default: wide(std::integral_constant<int, 1024>{}); break;
        }
      }
    } else if (K <= 20480) {
      // one lane per block: the workgroups are large enough as it is, and LDS (two rows per workgroup) bounds how
      // many a CU holds
      auto one_lane = [&](auto t_c) {
        constexpr int T = decltype(t_c)::value;
        if constexpr (NM ? T > 384 : !KP || T != 384)   // what two_lanes leaves
          launch_dma(reorder_quant_dma_kernel<32, T, kNS, IS_W, T, KP, NM, TI>, 32, kNS, T, kPerCu);
        else
          err = hipErrorInvalidValue;
      };
      switch (threads) {
        case 320: one_lane(std::integral_constant<int, 320>{}); break;
        case 384: one_lane(std::integral_constant<int, 384>{}); break;
        case 448: one_lane(std::integral_constant<int, 448>{}); break;
        case 512: one_lane(std::integral_constant<int, 512>{}); break;
        case 576: one_lane(std::integral_constant<int, 576>{}); break;
        default: one_lane(std::integral_constant<int, 640>{}); break;
      }
    } else {
      launch_dma(reorder_quant_dma_kernel<32, 0, 2, IS_W, 1024, KP, NM, TI>, 32, 2, threads, kPerCu);
    }
  };
  const std::true_type yes;
  const std::false_type no;
  if constexpr (IS_W) {
    if (src_rows != 0) dispatch(no, no, yes);
    else dispatch(no, no, no);
  } else {
    // Up to 16 rows, whose GEMMs take codes row by row and whose launch is all there is, nobody asks for their order: M = 8, N = 14336, K = 4096 with
    // RMSNorm 10.75 us instead of 10.85 (other widths go to few_rows).
    const bool decoded = gamma != nullptr && a_staged == 0 && rows <= 16 && K > 2048 && K <= 4096;
    if (gamma != nullptr && !decoded) dispatch(yes, yes, no);
    else if (keep_codes && !decoded) dispatch(yes, no, no);
    else if (!decoded) dispatch(no, no, no);
    else if (K <= 3072) launch_dma(reorder_quant_dma_kernel<16, 192, kNS, IS_W, 192, true, true, false, false>, 16, kNS, 192, kPerCu);
    else launch_dma(reorder_quant_dma_kernel<16, 256, kNS, IS_W, 256, true, true, false, false>, 16, kNS, 256, kPerCu);
  }
  return err;
}

template hipError_t launch_reorder_quant<false>(const void*, const int16_t*, int, int, int, int, int, uint8_t*, uint8_t*,
                                                uint8_t*, uint8_t*, uint8_t*, uint8_t*, const void*, float, bool, int, int, unsigned*, hipStream_t);
template hipError_t launch_reorder_quant<true>(const void*, const int16_t*, int, int, int, int, int, uint8_t*, uint8_t*,
                                               uint8_t*, uint8_t*, uint8_t*, uint8_t*, const void*, float, bool, int, int, unsigned*, hipStream_t);

}  // namespace mg
