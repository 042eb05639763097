// Mixed block-scaled GEMM on small workgroup tiles, 64 or 128 features x 64 or 128 tokens, for problems with too few tiles of
// 256 x 256 or 256 x 128 to fill the chip: waves that only copy and waves that only multiply.
//
// What bounded such launches on 256 x 128 tiles was not the memory (a tile alone on the chip took 0.30 us per stage of 128 K elements):
// a global -> LDS copy holds the wave that issues it for ~64 cycles (its addresses go out one per cycle; a CU accepts one
// from each of its SIMDs at a time, 1 KB per 16 cycles in all where it is put together from whole lines that are in the L2), so that waves that
// copy and multiply in turn leave the matrix cores idle.  Here four waves, one per SIMD, issue all copies, eight waves, two per SIMD, read
// fragments and multiply, and one barrier hands over WS stages at a time, each of them the work of 8 / WS of the math waves (fragments are read
// once per 2 x 2 tiles of 32 x 32 rather than once per 1 x 2).
// What bounds it now: with many stages the copies (M = 256, N = 4096, K = 14336: address unit busy 65 ... 69 % of the cycles, matrix cores 18 ... 21 %, the
// LDS's fragment reads 24 ... 28 %), with 32 stages latency as well (address unit 36 ... 51 %, waves waiting 52 ... 68 %; M = 1024, N = K = 4096: matrix
// cores 27 ... 32 %).  An instruction takes the address unit 19 ... 26 cycles with the tokens' codes stage by stage, 22 ... 32 row by row, of which 1 ... 11 and
// 10 ... 34 % are stalls on the cache behind it.  Clock stamps of an instrumented build, copies stage by stage of codes row by
// row: 64 x 64 tiles, K = 4096, one per CU: 270 cycles per stage, of which 64 are MFMAs' (150 without copies); a launch of them takes 1.2
// us until the first stages have landed, 2.7 us for 20 E2M1 and 1.3 for 12 later stages, 1.2 us to add the partial sums and store.
// Tile-major / row-major weights, of two or three layers in turn in the caches, before (skinny kernel or 256 x 128 tiles) -> now, us:
//   M = 256, N = 4096, K = 4096: 16.4 / 19.6 -> 8.3 / 8.6;   K = 14336: 45.6 / 59.9 -> 20.2 / 22.3
//   M = 512, N = 4096, K = 4096: 16.6 / 19.6 -> 10.0 / 12.0;  N = 1024, K = 8192: 27.6 / 34.8 -> 11.6 / 13.2
//   M = 64, N = 14336, K = 4096: 16.4 / 16.8 -> 8.8 / 9.3;   M = 128: 16.8 / 20.1 -> 10.1 / 12.3
//   M = 1024, N = 4096, K = 4096: 17.0 / 19.7 -> 14.5 / 16.5
// (from HBM: M = 256 10.6 / 10.8 and 30 / 30, M = 512 12.5 / 15.2 and 16.1 / 16.0, M = 64 13.7 / 14.1, M = 1024 17.6 / 19.2), all of these
// stage by stage on row-major codes; with batches copied as rows of their stages (BatchRow): K = 14336, M = 256 17.5 / 18.7;  M = 1024, K = 4096 12.6 / 13.1
// Tiles of 256 x 128 with the same division of work were level with the mixed waves of the 256 x 256 kernel (M = 2048, N =
// 4096, K = 12288: 57.6 against 56.3 us: 15 % fewer cycles at a clock as much lower; the chip is at its power limit there), tiles of
// 64 and 128 x 32 slower than 64 x 64 at every shape tried.
#include "mg_common.h"
#include "staged_codes.h"
#include "tile_order.h"

#include <type_traits>

namespace mg {

namespace {

constexpr int kCopyWaves = 4, kMathWaves = 8, kTileWaves = kCopyWaves + kMathWaves;
constexpr int kRingBytes = 156 * 1024;   // LDS for the ring of batches

typedef int v6i __attribute__((ext_vector_type(6)));
typedef uint16_t v8h __attribute__((ext_vector_type(8)));
typedef v8h v8h_any __attribute__((aligned(2)));

struct TileSeg {
  const uint8_t *a, *b, *sfa, *sfb;
  int blk;    // 32-element blocks
  int whole;  // whole 128-wide stages
};

struct TilePlan {
  TileSeg s4, s6, s8;
  int total;      // whole stages of all segments
  int N;          // weight rows
  int m_store;    // token rows that are stored
  int a_rows;     // token rows that may be read
  int a_staged;   // the token codes are stage by stage, of so many rows (0: row-major, see launch_reorder_quant)
  TileOrder order;   // workgroup -> tile
};

template <int FMT> struct Form;
template <> struct Form<kFmtE2M1> { static constexpr int row = 64; typedef v4i frag; };
template <> struct Form<kFmtE3M2> { static constexpr int row = 96; typedef v6i frag; };
template <> struct Form<kFmtE4M3> { static constexpr int row = 128; typedef v8i frag; };

__device__ __forceinline__ const uint8_t* uniform(const uint8_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<const uint8_t*>(((uint64_t)hi << 32) | lo);
}

// global[base + voff(lane)] -> LDS[lds_off + 16 * lane]; base and lds_off wave-uniform
__device__ __forceinline__ void copy_at(const uint8_t* base, unsigned voff, unsigned lds_off) {
  base = uniform(base);
  lds_off = __builtin_amdgcn_readfirstlane(lds_off);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               : : "v"(voff), "s"(base), "s"(lds_off) : "memory", "m0");
}
// the same with a 64-bit address per lane
__device__ __forceinline__ void copy_lane(const uint8_t* p, unsigned lds_off) {
  lds_off = __builtin_amdgcn_readfirstlane(lds_off);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(p), "s"(lds_off) : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
__device__ __forceinline__ void workgroup_barrier() { asm volatile("s_barrier" ::: "memory"); }
// the barriers of the last YOUNGER + 2 batches, with nothing more to issue; the last PARTIAL of them count for nothing
template <int YOUNGER, int PER, int PARTIAL>
__device__ __forceinline__ void drain() {
  wait_vm<(YOUNGER > PARTIAL ? YOUNGER - PARTIAL : 0) * PER>();
  workgroup_barrier();
  if constexpr (YOUNGER > 0) drain<YOUNGER - 1, PER, PARTIAL>();
  else workgroup_barrier();
}
// s_waitcnt lgkmcnt(0) that the compiler's own counting sees
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// Geometry of an instance.  TF x TT: the workgroup's tile; WT: tile-major weights; a batch of WS stages per barrier, each the
// work of 8 / WS math waves (WF along the features); ROWS: batches of one segment lie as rows of WS stages (BatchRow).
template <int TF_, int TT_, int WF_, int WS_, bool WT_, bool ROWS_>
struct Geo {
  static constexpr int TF = TF_, TT = TT_, WF = WF_, WS = WS_;
  static constexpr bool WT = WT_, ROWS = ROWS_;
  static constexpr int WM = kMathWaves / WF / WS;                          // math waves along tokens
  static constexpr int TN = TF / 32 / WF, TM = TT / 32 / WM;               // a wave's 32 x 32 tiles
  // a batch in LDS: per stage 1 KB of scales (32 pieces of the features, 32 of the tokens), then the weights, then the tokens
  static constexpr int kW = WS * 1024, kX = kW + WS * TF * 64;
  static constexpr int kBatch = kX + WS * TT * 128;
  static constexpr int NB = kRingBytes / kBatch < 8 ? kRingBytes / kBatch : 8;   // batches in the ring
  // the partial sums on their way out: per stage of a batch, fp32 rows of tokens
  static constexpr int kPitch = TF * 4 + 16, kPart = TT * kPitch;
  static_assert(WS > 1 && TN == 2 && (TM == 1 || TM == 2) && NB >= 3 && WS * kPart <= NB * kBatch, "tile geometry");
};

template <class G>
struct TileCtx {
  int lane, n0, m0;        // first feature, first token of the tile
  int last_col, last_row;  // last readable weight / token row, from the tile's first
};

// ---------------------------------------------------------------------------------------------
// Copies, dealt to the four copy waves.  A cache line is 128 bytes, a stage of a row of E2M1 codes 64, of E3M2 96: a batch whose stages are
// all of one segment is copied (and lies in LDS) as rows of WS stages, so that its lines are asked for once, in one piece (BatchRow).
// Stage by stage, every row's every line was fetched by two copies a batch or more apart: GEMM alone, tile-major / row-major weights,
// all E2M1, us: M = 256, N = 4096, K = 14336 17.2 -> 15.2 / - ; M = 512, N = 4096, K = 4096 8.9 -> 8.6 / 10.2 -> 8.7; M = 1024 11.9 -> 11.0 /
// 13.5 -> 11.1; M = 244, N = 12416, K = 13824, default plan - / 64.8 -> 48.3.  Short launches do not gain (batch_rows).
// A batch of two segments, and a last, partial one, go stage by stage: weights and E2M1 tokens 16 rows x 64 B per copy, the 16-byte
// pieces of row r permuted by XOR with r / 4, E3M2: rows of 96 B one after the other,
// their pieces rotated by one in rows 8 ... 15 of every 16: the 16 rows that a fragment read touches at a time lie on different
// banks (E3M2 rows as they are: 0.85 instead of 0.36 us per stage of 128 x 128).  E4M3 always goes stage by stage, a line per row: 8 rows x
// 128 B, permuted by XOR with r / 2.  Scales: the two atoms of 128 rows that hold the tile's rows, one copy per stage.
// Tile-major weights (16 KB per 256 features and stage: 1 KB per j = feature % 16, in it 64 bytes per feature / 16, even ones
// first): a copy takes what the tile's features have of 128 / TF blocks of 1 KB, whole lines, and row i of a 32-row fragment is the
// feature that WeightRows says.  (A workgroup has consecutive features: with whole 1 KB blocks, i.e. every other run of eight, two
// workgroups shared each line of the result: M = 1024, N = K = 4096 with the same operands in each launch 17.1 us, now 13.9; with one
// feature's 64 bytes per four lanes, half lines, M = 256, N = 4096, K = 14336 21.9 us, now 20.2.)
// ---------------------------------------------------------------------------------------------
// Rows of a weight fragment.  Row-major: row i of fragment T is feature 32 T + i of the tile, in copy block 2 T + i / 16.
// Tile-major, 128 features: copy block j / 2 holds [j % 2][feature / 16 % 2][feature / 32]; 64: j / 4 [j % 4][...][...].  Four
// consecutive rows of a fragment are four consecutive features, and the 16 rows read at a time (0-3, 12-15, 20-27 and the others)
// are four different feature / 16 with all four j % 4 each: with the pieces permuted by XOR with j, on different banks.
template <class G>
struct WeightRows {
  static __device__ __forceinline__ int feature(int T, int i) {
    if constexpr (!G::WT) return 32 * T + i;
    else if constexpr (G::TF == 128) return 16 * (2 * ((i >> 2) & 3) + (i >> 4)) + 4 * T + (i & 3);
    else return 16 * (2 * ((i >> 2) & 1) + ((i >> 3) & 1)) + 8 * T + 4 * (i >> 4) + (i & 3);
  }
  // of its 64 bytes in the stage's weights
  static __device__ __forceinline__ int lds(int T, int i) {
    if constexpr (!G::WT) return T * 2048 + i * 64;
    else if constexpr (G::TF == 128) return T * 2048 + ((i >> 1) & 1) * 1024 + (i & 1) * 512 + (i >> 4) * 256 + ((i >> 2) & 3) * 64;
    else return T * 2048 + (i >> 4) * 1024 + (i & 3) * 256 + ((i >> 3) & 1) * 128 + ((i >> 2) & 1) * 64;
  }
  // of its scale dword in the stage's scales; first: the tile's first feature in its atom of 128, / 32
  static __device__ __forceinline__ int scale(int T, int i, int first) {
    if constexpr (!G::WT) return i * 16 + ((first + T) & 3) * 4;
    else if constexpr (G::TF == 128) return T * 128 + (i >> 4) * 64 + (i & 3) * 16 + ((i >> 2) & 3) * 4;
    else return T * 256 + ((i >> 3) & 1) * 128 + (i >> 4) * 64 + (i & 3) * 16 + (first + ((i >> 2) & 1)) * 4;
  }
  // what a lane copies: the 16-byte piece of the atom (32 lanes) ...
  static __device__ __forceinline__ int scale_piece(int l) {
    if constexpr (!G::WT) return l;
    else if constexpr (G::TF == 128) return 16 * ((l >> 2) & 1) + 4 * (l >> 3) + (l & 3);
    else return 16 * ((l >> 3) & 1) + 8 * (l >> 4) + 4 * ((l >> 2) & 1) + (l & 3);
  }
  // ... and the offset of its 16 bytes of copy block b in the stage's 16 KB of tile-major weights
  static __device__ __forceinline__ unsigned tiled_offset(int b, int l, int n0) {
    const int j = G::TF == 128 ? 2 * b + (l >> 5) : 4 * b + (l >> 4);
    const int odd = G::TF == 128 ? (l >> 4) & 1 : (l >> 3) & 1, pair = G::TF == 128 ? (l >> 2) & 3 : (l >> 2) & 1;
    return (unsigned)(j * 1024 + (((n0 & 255) >> 5) + pair + 8 * odd) * 64 + (((l & 3) ^ (j & 3)) * 16));
  }
};

// n / P for a piece's number n < 2^15
template <int P>
__device__ __forceinline__ int row_of(int n) {
  static_assert(P == 8 || P == 16 || P == 6 || P == 12 || P == 24, "pieces per row");
  if constexpr ((P & (P - 1)) == 0) return n / P;
  else return (int)(__umul24((unsigned)n, 43691u) >> (P == 6 ? 18 : P == 12 ? 19 : 20));   // 43691 * 6 = 2^18 + 2
}

// Rows of a batch of one segment in LDS: BYTES per stage, WS stages, in 16-byte pieces; which piece lies where in its row depends on the
// row such that the 16 rows read at a time (see WeightRows) are on 16 different sixteenths of the 256 bytes of all banks: a power of two
// of pieces is permuted by XOR, 12 and 24 (E3M2) are rotated by as many steps as rows 12 and 24 pieces apart leave between them.
template <int BYTES, class G>
struct BatchRow {
  static constexpr int P = G::WS * BYTES / 16, bytes = 16 * P;
  static_assert(P == 8 || P == 12 || P == 16 || P == 24, "pieces per row");
  static __device__ __forceinline__ int key(int row) { return P == 16 ? row & 15 : P == 12 ? (row >> 2) & 3 : (row >> 1) & 7; }
  static __device__ __forceinline__ int place(int piece, int row) {   // of a piece in the row
    if constexpr ((P & (P - 1)) == 0) return piece ^ key(row);
    const int at = piece + key(row);
    return at >= P ? at - P : at;
  }
  static __device__ __forceinline__ int piece(int at, int row) {      // that lies there
    if constexpr ((P & (P - 1)) == 0) return at ^ key(row);
    const int p = at - key(row);
    return p < 0 ? p + P : p;
  }
};

template <int FMT, class G>
constexpr int kTokenCopiesAll = G::TT * Form<FMT>::row / 1024;   // per stage
// copies that every copy wave issues per whole batch, at least (a stage of a later segment has as many or more)
template <class G>
constexpr int kBatchCopies = G::WS * (G::TF / 64) + G::WS * kTokenCopiesAll<kFmtE2M1, G> / kCopyWaves + G::WS / kCopyWaves;

template <int FMT, class G>
struct SegCopy {
  static constexpr bool kRows = G::ROWS && FMT != kFmtE4M3;   // whole batches as rows of WS stages
  static constexpr int NW = G::TF / 64, NX = kTokenCopiesAll<FMT, G>, KX = (NX + kCopyWaves - 1) / kCopyWaves;
  static constexpr int BW = G::WS * NW, BX = G::WS * NX / kCopyWaves;   // of a whole batch
  static_assert(G::WS * NX % kCopyWaves == 0, "a batch's token copies are dealt evenly");
  typedef BatchRow<64, G> WRow;
  typedef BatchRow<kRows ? Form<FMT>::row : 64, G> XRow;
  const uint8_t *w, *x;         // bases of the next stage
  const uint8_t* sc;            // this lane's scale piece
  unsigned vw[NW], vx[KX], bw[BW], bx[BX];
  unsigned xstep;               // from a stage of the tokens to the next
  int wave;

  // token copies of a stage come in fours, a last pair is dealt to waves 0, 1 and 2, 3 in turn
  static_assert(NX % 2 == 0, "token copies in pairs");
  __device__ __forceinline__ int block(int k) const { return (k + 1) * kCopyWaves <= NX ? wave + kCopyWaves * k : (wave & 1) + kCopyWaves * k; }

  // the bases, and what batches copied as rows need
  __device__ __forceinline__ void init(const TileCtx<G>& c, const TileSeg& s, int a_staged, int wave_) {
    wave = wave_;
    const unsigned pitch = a_staged ? Form<FMT>::row : (unsigned)s.blk * (Form<FMT>::row / 4);
    xstep = a_staged ? (unsigned)a_staged * Form<FMT>::row : Form<FMT>::row;
    x = s.a + (size_t)c.m0 * pitch;
    if constexpr (G::WT) {
      w = s.b + (size_t)(c.n0 >> 8) * s.whole * 16384;
#pragma unroll
      for (int k = 0; k < NW; ++k) vw[k] = WeightRows<G>::tiled_offset(wave + kCopyWaves * k, c.lane, c.n0);
    } else {
      w = s.b + (size_t)c.n0 * s.blk * 16;
      if constexpr (kRows) {
#pragma unroll
        for (int k = 0; k < BW; ++k) {
          const int chunk = 64 * (wave + kCopyWaves * k) + c.lane, row = row_of<WRow::P>(chunk);
          bw[k] = __umul24(min(row, c.last_col), 16 * s.blk) + WRow::piece(chunk - row * WRow::P, row) * 16;
        }
      }
    }
    if constexpr (kRows) {
#pragma unroll
      for (int k = 0; k < BX; ++k) {
        const int chunk = 64 * (wave + kCopyWaves * k) + c.lane, row = row_of<XRow::P>(chunk);
        bx[k] = __umul24(min(row, c.last_row), pitch) + XRow::piece(chunk - row * XRow::P, row) * 16;
      }
    }
    const int katoms = (s.blk + 3) >> 2;
    const uint8_t* const of_features = s.sfb + (size_t)(c.n0 >> 7) * katoms * 512;
    const uint8_t* const of_rows = s.sfa + (size_t)(c.m0 >> 7) * katoms * 512;
    sc = c.lane < 32 ? of_features + WeightRows<G>::scale_piece(c.lane) * 16 : of_rows + (c.lane & 31) * 16;
  }
  // what single stages need
  __device__ __forceinline__ void init_stages(const TileCtx<G>& c, const TileSeg& s, int a_staged) {
    const int r = c.lane >> 2, p = (c.lane & 3) ^ ((c.lane >> 4) & 3);
    if constexpr (!G::WT) {
#pragma unroll
      for (int k = 0; k < NW; ++k) vw[k] = __umul24(min(16 * (wave + kCopyWaves * k) + r, c.last_col), 16 * s.blk) + p * 16;
    }
    const unsigned pitch = a_staged ? Form<FMT>::row : (unsigned)s.blk * (Form<FMT>::row / 4);
#pragma unroll
    for (int k = 0; k < KX; ++k) {
      const int b = block(k);
      if constexpr (FMT == kFmtE2M1) {
        vx[k] = __umul24(min(16 * b + r, c.last_row), pitch) + p * 16;
      } else if constexpr (FMT == kFmtE3M2) {   // the pieces of rows 8 ... 15 of every 16 rotated by one
        const int chunk = 64 * b + c.lane, row = row_of<6>(chunk), at = chunk - row * 6;
        const int piece = (row & 8) ? (at == 0 ? 5 : at - 1) : at;
        vx[k] = __umul24(min(row, c.last_row), pitch) + piece * 16;
      } else {
        const int row = 8 * b + (c.lane >> 3);
        vx[k] = __umul24(min(row, c.last_row), pitch) + (((c.lane & 7) ^ ((row >> 1) & 7)) * 16);
      }
    }
  }

  // What does not divide by the copy waves goes to other ones in every stage (t: of all stages).
  __device__ __forceinline__ void scales(int t, unsigned at) {
    const int turn = 2 * (~t & 1) + ((t >> 1) & 1);   // every wave once in four stages
    if (turn == wave) copy_lane(sc, at);
    sc += 512;
  }
  // the next stage, t-th of all, as stage u of a batch
  __device__ __forceinline__ void issue(int t, int u, unsigned batch) {
#pragma unroll
    for (int k = 0; k < NW; ++k) copy_at(w, vw[k], batch + G::kW + G::TF * 64u * u + 1024u * (wave + kCopyWaves * k));
#pragma unroll
    for (int k = 0; k < KX; ++k)
      if ((k + 1) * kCopyWaves <= NX || (wave >> 1) == (t & 1)) copy_at(x, vx[k], batch + G::kX + G::TT * 128u * u + 1024u * block(k));
    scales(t, batch + 1024u * u);
    w += G::WT ? 16384 : 64;
    x += xstep;
  }
  // the next WS stages
  __device__ __forceinline__ void issue_batch(int t, unsigned batch) {
    if constexpr (!kRows) {
#pragma unroll
      for (int u = 0; u < G::WS; ++u) issue(t + u, u, batch);
    } else {
      if constexpr (G::WT) {
#pragma unroll
        for (int u = 0; u < G::WS; ++u)
#pragma unroll
          for (int k = 0; k < NW; ++k) copy_at(w + u * 16384, vw[k], batch + G::kW + G::TF * 64u * u + 1024u * (wave + kCopyWaves * k));
      } else {
#pragma unroll
        for (int k = 0; k < BW; ++k) copy_at(w, bw[k], batch + G::kW + 1024u * (wave + kCopyWaves * k));
      }
#pragma unroll
      for (int k = 0; k < BX; ++k) copy_at(x, bx[k], batch + G::kX + 1024u * (wave + kCopyWaves * k));
#pragma unroll
      for (int u = 0; u < G::WS; ++u) scales(t + u, batch + 1024u * u);
      w += G::WS * (G::WT ? 16384 : 64);
      x += G::WS * Form<FMT>::row;
    }
  }
};

// ---------------------------------------------------------------------------------------------
// Fragments of one 64-wide K half
// ---------------------------------------------------------------------------------------------
template <int FMT, class G>
struct TileFrags {
  v4i w[G::TN];
  typename Form<FMT>::frag x[G::TM];
};

// Per-lane offsets inside a batch of what a wave reads of its stage; [..][H]: of K half H.  Rows of WS stages (ROWS) or of one.
struct ReadAt {
  int w[2], x[2], h[2];   // 16-byte pieces of weights and tokens, 8-byte ones of E3M2 tokens (E4M3: x[H] and, 32 bytes off under XOR, h[H])
};
template <int FMT, bool ROWS, class G>
__device__ __forceinline__ ReadAt read_at(int i, int g, int wf, int wm, int ws) {
  ReadAt at;
  const int T0 = wf * G::TN, row0 = wm * G::TM * 32;
#pragma unroll
  for (int H = 0; H < 2; ++H) {
    if constexpr (ROWS && !G::WT) {
      typedef BatchRow<64, G> Row;
      at.w[H] = G::kW + (T0 * 32 + i) * Row::bytes + Row::place(4 * ws + 2 * H + g, i) * 16;
    } else {
      at.w[H] = G::kW + ws * G::TF * 64 + WeightRows<G>::lds(T0, i) + (((2 * H + g) ^ (G::WT ? i & 3 : (i >> 2) & 3)) * 16);
    }
    if constexpr (ROWS) {
      typedef BatchRow<Form<FMT>::row, G> Row;
      const int x = G::kX + (row0 + i) * Row::bytes;
      if constexpr (FMT == kFmtE2M1) {
        at.x[H] = x + Row::place(4 * ws + 2 * H + g, i) * 16;
        at.h[H] = 0;
      } else {   // block 2H is piece 3H and the first half of piece 3H + 1, block 2H + 1 the other half and piece 3H + 2
        at.x[H] = x + Row::place(6 * ws + 3 * H + 2 * g, i) * 16;
        at.h[H] = x + Row::place(6 * ws + 3 * H + 1, i) * 16 + 8 * g;
      }
    } else {
      const int x = G::kX + ws * G::TT * 128 + (row0 + i) * Form<FMT>::row;
      if constexpr (FMT == kFmtE2M1) {
        at.x[H] = x + (((2 * H + g) ^ ((i >> 2) & 3)) * 16);
        at.h[H] = 0;
      } else if constexpr (FMT == kFmtE3M2) {
        const int turn = (i >> 3) & 1;
        auto piece = [&](int p) { return (p + turn == 6 ? 0 : p + turn) * 16; };
        at.x[H] = x + piece(3 * H + 2 * g);
        at.h[H] = x + piece(3 * H + 1) + 8 * g;
      } else {   // K [16g, 16g+16) and [32+16g, ...) of the half
        at.x[H] = x + (((4 * H + g) ^ ((i >> 1) & 7)) * 16);
        at.h[H] = x + (((4 * H + 2 + g) ^ ((i >> 1) & 7)) * 16);
      }
    }
  }
  return at;
}

__device__ __forceinline__ v8i widened(v4i v) { return __builtin_shufflevector(v, v, 0, 1, 2, 3, -1, -1, -1, -1); }
__device__ __forceinline__ v8i widened(v6i v) { return __builtin_shufflevector(v, v, 0, 1, 2, 3, 4, 5, -1, -1); }
__device__ __forceinline__ v8i widened(v8i v) { return v; }

template <int FMT, int H, bool ROWS, class G>
__device__ __forceinline__ void read_half(TileFrags<FMT, G>& f, const uint8_t* batch, const ReadAt& r, int g) {
  constexpr int kWTile = ROWS && !G::WT ? 32 * BatchRow<64, G>::bytes : 2048;
  constexpr int kXTile = 32 * Form<FMT>::row * (ROWS ? G::WS : 1);
#pragma unroll
  for (int t = 0; t < G::TN; ++t) f.w[t] = *reinterpret_cast<const v4i*>(batch + r.w[H] + t * kWTile);
#pragma unroll
  for (int t = 0; t < G::TM; ++t) {
    const v4i a = *reinterpret_cast<const v4i*>(batch + r.x[H] + t * kXTile);
    if constexpr (FMT == kFmtE2M1) {
      f.x[t] = a;
    } else if constexpr (FMT == kFmtE3M2) {
      const v2i b = *reinterpret_cast<const v2i*>(batch + r.h[H] + t * kXTile);
      f.x[t] = g ? v6i{b[0], b[1], a[0], a[1], a[2], a[3]} : v6i{a[0], a[1], a[2], a[3], b[0], b[1]};
    } else {
      const v4i b = *reinterpret_cast<const v4i*>(batch + r.h[H] + t * kXTile);
      f.x[t] = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
}

template <class G>
struct TileScales {
  int w[G::TN], x[G::TM];
};
// Scale dwords of the wave's fragments in a stage.  Of two fragments the lower 32 lanes read the first one's and the upper
// ones the second one's (a dword read occupies the LDS for as long as a 16-byte one).
template <class G>
struct RawScales {
  int w, x;
};
template <class G>
__device__ __forceinline__ void read_scales(RawScales<G>& s, const uint8_t* batch, int sw, int sx) {
  s.w = *reinterpret_cast<const int*>(batch + sw);
  s.x = *reinterpret_cast<const int*>(batch + sx);
}
__device__ __forceinline__ void both_halves(int v, int& lower, int& upper) {
  const auto p = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
  lower = (int)p[0];   // the lower lanes' value in all lanes
  upper = (int)p[1];
}
template <class G>
__device__ __forceinline__ TileScales<G> shifted(const RawScales<G>& s, int g) {
  TileScales<G> o;
  both_halves(s.w, o.w[0], o.w[1]);
  if constexpr (G::TM == 2) both_halves(s.x, o.x[0], o.x[1]);
  else o.x[0] = s.x;
#pragma unroll
  for (int t = 0; t < G::TN; ++t) o.w[t] = (int)((unsigned)o.w[t] >> (8 * g));
#pragma unroll
  for (int t = 0; t < G::TM; ++t) o.x[t] = (int)((unsigned)o.x[t] >> (8 * g));
  return o;
}

// MFMAs [M0, M1) of a K half
template <int FMT, int H, class G, int M0, int M1>
__device__ __forceinline__ void multiply(v16f (&acc)[G::TN][G::TM], const TileFrags<FMT, G>& f, const TileScales<G>& sc) {
#pragma unroll
  for (int k = M0; k < M1; ++k) {
    const int tn = k / G::TM, tm = k % G::TM;
    acc[tn][tm] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(widened(f.w[tn]), widened(f.x[tm]), acc[tn][tm], kFmtE2M1, FMT, 2 * H, sc.w[tn],
                                                                  2 * H, sc.x[tm]);
  }
}

// The 0 ... 3 blocks of 32 a segment has beyond its whole stages, straight from global memory, before the K loop; each segment's
// by the waves of another stage of the batch.
template <int FMT, class G>
struct Rest {
  TileFrags<FMT, G> f;
  TileScales<G> sc;
};
template <int FMT, int H, class G>
__device__ __forceinline__ void rest_load(Rest<FMT, G>& r, const TileCtx<G>& c, const TileSeg& s, int N, int a_staged, int wf, int wm) {
  const int rem = s.blk & 3;
  const int i = c.lane & 31, g = c.lane >> 5, q = s.blk >> 2, katoms = (s.blk + 3) >> 2;
  const int kb = 4 * q + min(2 * H + g, rem - 1), kb0 = 4 * q + 2 * H, kb1 = 4 * q + min(2 * H + 1, rem - 1);   // blocks that exist
#pragma unroll
  for (int t = 0; t < G::TN; ++t) {
    const int n = c.n0 + min(WeightRows<G>::feature(wf * G::TN + t, i), c.last_col);
    const uint8_t* p = G::WT ? s.b + (size_t)(N >> 8) * q * 16384 + ((size_t)n * rem + (kb - 4 * q)) * 16 : s.b + ((size_t)n * s.blk + kb) * 16;
    r.f.w[t] = *reinterpret_cast<const v4i*>(p);
    r.sc.w[t] = s.sfb[sf_offset(n, kb, katoms)];
  }
#pragma unroll
  for (int t = 0; t < G::TM; ++t) {
    const int m = c.m0 + min((wm * G::TM + t) * 32 + i, c.last_row);
    // (behind codes that are stage by stage: rows of the rem blocks; row points to where the row's first block would be)
    const uint8_t* row = a_staged ? s.a + (size_t)a_staged * q * Form<FMT>::row + (size_t)m * rem * (Form<FMT>::row / 4) - (size_t)q * Form<FMT>::row
                                  : s.a + (size_t)m * s.blk * (Form<FMT>::row / 4);
    r.sc.x[t] = s.sfa[sf_offset(m, kb, katoms)];
    if constexpr (FMT == kFmtE2M1) {
      r.f.x[t] = *reinterpret_cast<const v4i*>(row + (size_t)kb * 16);
    } else if constexpr (FMT == kFmtE3M2) {
      const v2i* v = reinterpret_cast<const v2i*>(row + (size_t)kb * 24);
      const v2i a = v[0], b = v[1], e = v[2];
      r.f.x[t] = v6i{a[0], a[1], b[0], b[1], e[0], e[1]};
    } else {
      const v4i a = *reinterpret_cast<const v4i*>(row + (size_t)kb0 * 32 + g * 16), b = *reinterpret_cast<const v4i*>(row + (size_t)kb1 * 32 + g * 16);
      r.f.x[t] = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
}
// what lies past the segment's end is zero
template <int FMT, int H, class G>
__device__ __forceinline__ void rest_multiply(v16f (&acc)[G::TN][G::TM], Rest<FMT, G>& r, const TileSeg& s, int g) {
  const int rem = s.blk & 3;
  const bool ok = 2 * H + g < rem, ok1 = 2 * H + 1 < rem;
#pragma unroll
  for (int t = 0; t < G::TN; ++t) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r.f.w[t][e] = ok ? r.f.w[t][e] : 0;
    r.sc.w[t] = ok ? r.sc.w[t] : 127;
  }
#pragma unroll
  for (int t = 0; t < G::TM; ++t) {
    r.sc.x[t] = ok ? r.sc.x[t] : 127;
    if constexpr (FMT == kFmtE4M3) {
#pragma unroll
      for (int e = 4; e < 8; ++e) r.f.x[t][e] = ok1 ? r.f.x[t][e] : 0;
    } else {
#pragma unroll
      for (int e = 0; e < (FMT == kFmtE2M1 ? 4 : 6); ++e) r.f.x[t][e] = ok ? r.f.x[t][e] : 0;
    }
  }
  multiply<FMT, 0, G, 0, G::TN * G::TM>(acc, r.f, r.sc);
}
template <int H, class G>
__device__ __forceinline__ void rest_half(v16f (&acc)[G::TN][G::TM], const TileCtx<G>& c, const TilePlan& p, int wf, int wm, int ws, int g) {
  const bool has4 = (p.s4.blk & 3) > 2 * H && ws == 1 % G::WS, has6 = (p.s6.blk & 3) > 2 * H && ws == 2 % G::WS,
             has8 = (p.s8.blk & 3) > 2 * H && ws == 3 % G::WS;   // wave-uniform
  Rest<kFmtE2M1, G> r4;
  Rest<kFmtE3M2, G> r6;
  Rest<kFmtE4M3, G> r8;
  if (has4) rest_load<kFmtE2M1, H, G>(r4, c, p.s4, p.N, p.a_staged, wf, wm);
  if (has6) rest_load<kFmtE3M2, H, G>(r6, c, p.s6, p.N, p.a_staged, wf, wm);
  if (has8) rest_load<kFmtE4M3, H, G>(r8, c, p.s8, p.N, p.a_staged, wf, wm);
  __builtin_amdgcn_sched_barrier(0);
  if (has4) rest_multiply<kFmtE2M1, H, G>(acc, r4, p.s4, g);
  if (has6) rest_multiply<kFmtE3M2, H, G>(acc, r6, p.s6, g);
  if (has8) rest_multiply<kFmtE4M3, H, G>(acc, r8, p.s8, g);
}

// All arguments into scalar registers in one batch of loads: fetched where they are first used they cost a round trip to the
// argument buffer each time, before the first copy goes out.
__device__ __forceinline__ void pin_plan(const TilePlan& p, const Epilogue& ep, const uint16_t* d) {
  asm volatile("" : : "s"(p.s4.a), "s"(p.s4.b), "s"(p.s4.sfa), "s"(p.s4.sfb), "s"(p.s4.blk), "s"(p.s4.whole), "s"(p.s6.a), "s"(p.s6.b),
               "s"(p.s6.sfa), "s"(p.s6.sfb), "s"(p.s6.blk), "s"(p.s6.whole), "s"(p.s8.a), "s"(p.s8.b), "s"(p.s8.sfa), "s"(p.s8.sfb),
               "s"(p.s8.blk), "s"(p.s8.whole), "s"(p.total), "s"(p.N), "s"(p.m_store), "s"(p.a_rows), "s"(p.a_staged), "s"(p.order.xlog), "s"(p.order.div),
               "s"(p.order.div2), "s"(p.order.magic), "s"(p.order.grid_x), "s"(p.order.tiles), "s"(ep.bias), "s"(ep.n_out), "s"(d));
}

template <int TF, int TT, int WF, int WS, bool WT, bool REM, bool ROWS>
__global__ void __launch_bounds__(64 * kTileWaves)
mixed_gemm_tile_kernel(TilePlan plan, Epilogue ep, uint16_t* __restrict__ d) {
  typedef Geo<TF, TT, WF, WS, WT, ROWS> G;
  constexpr int NB = G::NB;
  extern __shared__ __align__(16) uint8_t lds[];
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  pin_plan(plan, ep, d);
  const int wg = blockIdx.y * plan.order.grid_x + blockIdx.x;
  if (wg >= plan.order.tiles) return;   // (the last row of a grid of several)
  int tn, tm;
  tile_at(plan.order, wg, tn, tm);
  TileCtx<G> c;
  c.lane = threadIdx.x & 63;
  c.n0 = tn * TF;
  c.m0 = tm * TT;
  c.last_col = min(plan.N - c.n0, TF) - 1;
  c.last_row = min(plan.a_rows - c.m0, TT) - 1;
  const int total = plan.total, t6 = plan.s4.whole, t8 = t6 + plan.s6.whole, batches = (total + WS - 1) / WS;

  if (wave < kCopyWaves) {
    // ------------------------------------------------------------------ copy waves
    SegCopy<kFmtE2M1, G> k4;
    SegCopy<kFmtE3M2, G> k6;
    SegCopy<kFmtE4M3, G> k8;
    unsigned batch = lds0;
    const unsigned ring_end = lds0 + NB * G::kBatch;
    auto advance = [&]() __attribute__((always_inline)) {
      batch += G::kBatch;
      batch = batch == ring_end ? lds0 : batch;
    };
    // The first NB batches at once, then one more behind each barrier.  Before the barrier that hands over a batch, all but
    // the copies of the NB - 2 younger ones have landed (kBatchCopies each at least; a last, partial one is counted as none).
    constexpr int LB = kBatchCopies<G>;
    // whole batches of one segment that end by stage `last`
    auto whole = [&](auto& k, int& t, int last) __attribute__((always_inline)) {
      for (; t + WS <= last; t += WS) {
        k.issue_batch(t, batch);
        advance();
      }
    };
    // the same behind a barrier each
    auto stream = [&](auto& k, int& t, int last) __attribute__((always_inline)) {
      for (; t + WS <= last; t += WS) {
        wait_vm<(NB - 2) * LB>();
        workgroup_barrier();
        k.issue_batch(t, batch);
        advance();
      }
    };
    // stages up to `last`, whatever their segments, one by one: whole batches but for the last one of all
    auto one_by_one = [&](int& t, int last) __attribute__((always_inline)) {
      auto stages = [&](auto& k, int end) __attribute__((always_inline)) {
        for (; t < end; ++t) {
          k.issue(t, t % WS, batch);
          if (t % WS == WS - 1) advance();
        }
      };
      stages(k4, min(last, t6));
      stages(k6, min(last, t8));
      stages(k8, last);
    };
    // batches up to stage `last` (a whole number of them, or all), whatever their segments
    auto fill = [&](int& t, int last) __attribute__((always_inline)) {
      if constexpr (!ROWS) {
        one_by_one(t, last);
      } else {
        whole(k4, t, min(last, t6));
        if (t < t6 && t < last) one_by_one(t, min(last, t + WS));
        whole(k6, t, min(last, t8));
        if (t < t8 && t < last) one_by_one(t, min(last, t + WS));
        whole(k8, t, last);
        if (t < last) one_by_one(t, last);
      }
    };
    int t = 0;
    constexpr int kFirst = NB * WS;
    const int a_staged = ROWS ? 0 : plan.a_staged;
    auto init_rest = [&]() __attribute__((always_inline)) {
      if (ROWS && t6 % WS) k4.init_stages(c, plan.s4, a_staged);
      k6.init(c, plan.s6, a_staged, wave);
      if (!ROWS || t6 % WS || t8 % WS) k6.init_stages(c, plan.s6, a_staged);
      k8.init(c, plan.s8, a_staged, wave);
      k8.init_stages(c, plan.s8, a_staged);
    };
    k4.init(c, plan.s4, a_staged, wave);
    if constexpr (!ROWS) k4.init_stages(c, plan.s4, a_staged);
    const bool short4 = t6 < kFirst;
    if (short4) init_rest();
    if (ROWS || total >= kFirst) {   // (batch_rows)
      // two batches, then the multiplying starts on the first of them, then the rest of the ring
      fill(t, 2 * WS);
      wait_vm<LB>();
      workgroup_barrier();   // batch 0 has landed
      fill(t, kFirst);
      if (!short4) init_rest();
      stream(k4, t, t6);
      if (t < t6 && t + WS <= total) {   // a batch of two or three segments
        wait_vm<(NB - 2) * LB>();
        workgroup_barrier();
        one_by_one(t, t + WS);
      }
      stream(k6, t, t8);
      if (t < t8 && t + WS <= total) {
        wait_vm<(NB - 2) * LB>();
        workgroup_barrier();
        one_by_one(t, t + WS);
      }
      stream(k8, t, total);
      if (t < total) {   // the last, partial batch
        wait_vm<(NB - 2) * LB>();
        workgroup_barrier();
        one_by_one(t, total);
        drain<NB - 2, LB, 1>();
      } else {
        drain<NB - 2, LB, 0>();
      }
    } else {   // all of them at once
      fill(t, total);
      wait_vm<0>();
      for (int q = 0; q <= batches; ++q) workgroup_barrier();
    }
  } else {
    // ------------------------------------------------------------------ math waves
    const int mw = wave - kCopyWaves, wf = mw % WF, wm = (mw / WF) % G::WM, ws = mw / (WF * G::WM);
    const int i = c.lane & 31, g = c.lane >> 5;
    const int sw = ws * 1024 + WeightRows<G>::scale(wf * G::TN + g, i, (c.n0 & 127) >> 5);
    const int sx = ws * 1024 + 512 + i * 16 + (((c.m0 & 127) >> 5) + wm * G::TM + (G::TM == 2 ? g : 0)) * 4;

    v16f acc[G::TN][G::TM];
#pragma unroll
    for (int a = 0; a < G::TN; ++a)
#pragma unroll
      for (int b = 0; b < G::TM; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
    if constexpr (REM) {
      rest_half<0, G>(acc, c, plan, wf, wm, ws, g);
      rest_half<1, G>(acc, c, plan, wf, wm, ws, g);
    }
    workgroup_barrier();   // batch 0 has landed
    const uint8_t* batch = lds;
    const uint8_t* const ring_end = lds + NB * G::kBatch;
    auto next_batch = [&]() __attribute__((always_inline)) {
      batch += G::kBatch;
      batch = batch == ring_end ? lds : batch;
    };
    // This wave's stages of `stages` batches, all of one format.  Everything between two barriers is one basic block with its order fixed by
    // scheduling barriers: an MFMA, the reads of the next half, the other MFMAs (the compiler would sink them behind the barrier).
    auto run = [&](auto fmt_c, auto rows_c, int stages) __attribute__((always_inline)) {
      constexpr int FMT = decltype(fmt_c)::value;
      constexpr bool BY_ROWS = decltype(rows_c)::value, RUN = BY_ROWS || FMT == kFmtE4M3 || !ROWS;
      if (stages == 0) return;
      int row = i;
      asm volatile("" : "+v"(row));   // the addresses of this format only: those of all five would be kept from the start
      const ReadAt at = read_at<FMT, BY_ROWS, G>(row, g, wf, wm, ws);
      TileFrags<FMT, G> fa, fb, fn;
      RawScales<G> raw;
      TileScales<G> sc;
      read_scales<G>(raw, batch, sw, sx);
      read_half<FMT, 0, BY_ROWS, G>(fa, batch, at, g);
      auto first_half = [&]() __attribute__((always_inline)) {
        wait_lds();
        sc = shifted<G>(raw, g);
        multiply<FMT, 0, G, 0, 1>(acc, fa, sc);
        __builtin_amdgcn_sched_barrier(0);
        read_half<FMT, 1, BY_ROWS, G>(fb, batch, at, g);
        __builtin_amdgcn_sched_barrier(0);
        multiply<FMT, 0, G, 1, G::TN * G::TM>(acc, fa, sc);
        __builtin_amdgcn_sched_barrier(0);
        wait_lds();
        workgroup_barrier();   // the next batch has landed; this one is in registers
        next_batch();
        __builtin_amdgcn_sched_barrier(0);
        multiply<FMT, 1, G, 0, 1>(acc, fb, sc);
        __builtin_amdgcn_sched_barrier(0);
      };
      if constexpr (RUN) {
        for (int q = 1; q < stages; ++q) {
          first_half();
          read_scales<G>(raw, batch, sw, sx);
          read_half<FMT, 0, BY_ROWS, G>(fn, batch, at, g);
          __builtin_amdgcn_sched_barrier(0);
          multiply<FMT, 1, G, 1, G::TN * G::TM>(acc, fb, sc);
          __builtin_amdgcn_sched_barrier(0);
          fa = fn;
        }
      }   // (else a single stage)
      first_half();
      multiply<FMT, 1, G, 1, G::TN * G::TM>(acc, fb, sc);
    };
    const std::integral_constant<int, kFmtE2M1> f4;
    const std::integral_constant<int, kFmtE3M2> f6;
    const std::integral_constant<int, kFmtE4M3> f8;
    const std::true_type rows;
    const std::false_type single;
    // Batches [0, e4) are all E2M1, [b6, e6) all E3M2; e4 if it is below b6 has stages of several segments, and so has e6 where E3M2
    // ends inside it.  (E4M3 stages are the last of every wave.)
    const int e4 = t6 / WS, b6 = (t6 + WS - 1) / WS, e6 = max(t8 / WS, b6);
    auto mine = [&](int t) { return (max(t - ws, 0) + WS - 1) / WS; };   // of the first t stages
    const int first = e4 * WS + ws, second = e6 * WS + ws;
    if constexpr (ROWS) {
      run(f4, rows, e4);
      run(f4, single, first < t6);
      run(f6, single, e4 < b6 && first >= t6 && first < t8);
      run(f6, rows, e6 - b6);
      run(f6, single, second < t8);
    } else {
      run(f4, single, mine(t6));
      run(f6, single, mine(t8) - mine(t6));
    }
    run(f8, single, mine(total) - mine(t8));
    if (mine(total) < batches) workgroup_barrier();

    // Nothing reads or fills the ring any more.  The partial sums to LDS, as rows of tokens: a lane holds token i of its 32 x 32
    // tiles and fragment rows 8 (v / 4) + 4 g + v % 4, four consecutive features at a time.
#pragma unroll
    for (int b = 0; b < G::TM; ++b) {
      uint8_t* row = lds + ws * G::kPart + ((wm * G::TM + b) * 32 + i) * G::kPitch;
#pragma unroll
      for (int a = 0; a < G::TN; ++a)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq)
          *reinterpret_cast<v4f*>(row + WeightRows<G>::feature(wf * G::TN + a, 8 * vq + 4 * g) * 4) =
              v4f{acc[a][b][4 * vq], acc[a][b][4 * vq + 1], acc[a][b][4 * vq + 2], acc[a][b][4 * vq + 3]};
    }
    wait_lds();
  }
  workgroup_barrier();

  // All waves add the partial sums of a batch's stages, in their order, and store pieces of eight features.
  {
    constexpr int PR = TF / 8, RI = 64 / PR;   // pieces per row, rows per instruction
    const int piece = c.lane % PR, sub = c.lane / PR, col = c.n0 + piece * 8;
    const int n_out = ep.n_out, cols_left = n_out - col;
    v8h bias = {};
    if (ep.bias != nullptr) {   // wave-uniform
#pragma unroll
      for (int e = 0; e < 8; ++e) bias[e] = e < cols_left ? ep.bias[col + e] : (uint16_t)0;
    }
    const bool aligned = (n_out & 7) == 0;
    for (int r0 = wave * RI; r0 < TT; r0 += kTileWaves * RI) {
      const int r = r0 + sub, m = c.m0 + r;
      if (r >= TT || m >= plan.m_store || cols_left <= 0) continue;
      v8h h;
      const uint8_t* at = lds + r * G::kPitch + piece * 32;
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        v4f sum = *reinterpret_cast<const v4f*>(at + 4 * e);
#pragma unroll
        for (int o = 1; o < WS; ++o) sum += *reinterpret_cast<const v4f*>(at + o * G::kPart + 4 * e);
#pragma unroll
        for (int x = 0; x < 4; ++x) h[e + x] = __builtin_bit_cast(uint16_t, (__bf16)sum[x]);
      }
      if (ep.bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = add_bf16(h[e], bias[e]);
      }
      uint16_t* dst = d + (size_t)m * n_out + col;
      if (cols_left >= 8) {
        if (aligned) __builtin_nontemporal_store(h, reinterpret_cast<v8h*>(dst));
        else __builtin_nontemporal_store(h, reinterpret_cast<v8h_any*>(dst));
      } else {
#pragma unroll
        for (int e = 0; e < 7; ++e)
          if (e < cols_left) dst[e] = h[e];
      }
    }
  }
}

// Whether batches of one segment are copied as rows of WS stages.  The lines it saves against what it costs once (more offsets before the
// first copies, batches that are not whole in code of their own): one by one / as rows, us, tile-major, row-major weights, default plan:
//   64 x 64, M = 256, N = 4096: 16 stages 5.53 / 6.03, 5.45 / 6.02; 28 7.36 / 7.44, 7.78 / 7.66; 32 8.06 / 7.81, 8.47 / 8.07; 64 12.5 / 11.1;
//     112 19.8 / 17.5, 22.3 / 18.7
//   128 x 64, M = 512: 8 stages 5.30 / 5.72, 5.43 / 5.83; 16 6.63 / 7.00, 7.24 / 7.19; 32 9.52 / 9.47, 11.5 / 10.1; 48 13.9 / 14.1; 64 15.3 / 14.4
//     (its weights are most of its bytes: whole lines already where they are tile-major)
//   128 x 128, M = 1024: 8 stages 6.77 / 7.12, 7.11 / 7.36; 16 9.24 / 9.10, 10.1 / 9.24; 32 13.7 / 12.6, 15.4 / 13.1; 48 20.6 / 19.8
// (Least where a row of codes is not whole lines, K = 3072 and 5120: there the stages of a batch still end in the middle of one.)
constexpr bool batch_rows(int tf, int tt, bool w_tiled, int stages) {
  return stages >= (tf == 64 ? 32 : tt == 64 && w_tiled ? 56 : 16);
}

template <int TF, int TT, int WF, int WS>
hipError_t launch_geo(const TilePlan& p, bool w_tiled, bool rem, const Epilogue& ep, uint16_t* d, hipStream_t stream) {
  auto of = [&](auto rows_c) {
    constexpr bool ROWS = decltype(rows_c)::value;
    return w_tiled ? (rem ? mixed_gemm_tile_kernel<TF, TT, WF, WS, true, true, ROWS> : mixed_gemm_tile_kernel<TF, TT, WF, WS, true, false, ROWS>)
                   : (rem ? mixed_gemm_tile_kernel<TF, TT, WF, WS, false, true, ROWS> : mixed_gemm_tile_kernel<TF, TT, WF, WS, false, false, ROWS>);
  };
  // (codes that are stage by stage are whole lines as they are)
  const auto kernel = p.a_staged == 0 && batch_rows(TF, TT, w_tiled, p.total) ? of(std::true_type()) : of(std::false_type());
  static_assert((int64_t)kMostTilesAcross * 64 * kTileWaves < (int64_t)1 << 32, "threads along a dimension of the grid");
  typedef Geo<TF, TT, WF, WS, false, false> G;
  constexpr int kLds = G::NB * G::kBatch;
  static_assert(!batch_rows(TF, TT, false, G::NB * WS - 1) && !batch_rows(TF, TT, true, G::NB * WS - 1), "with rows the ring is filled at least once");
  if (hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds); e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(p.order.grid_x, grid_rows(p.order)), dim3(64 * kTileWaves), kLds, stream, p, ep, d);
  return hipGetLastError();
}

}  // namespace

struct TilePlanChoice { int tf, tt; double us; };

// The tile with the lowest estimate.  A workgroup has its CU to itself (LDS), so a launch is rounds of them; microseconds: fixed,
// per round, per stage and round, per stage with all CUs busy, per MB of results, per round with blocks past the whole stages.
// Fitted to 450 measured calls each (17 ... 2600 tokens, N 384 ... 28672, K 1024 ... 18944, tile-major weights; rms error 10 %,
// before the runs of tiles per XCD of tile_order.h, which made launches of other than 8 n tiles up to 1.4 times as fast):
// the tile taken is in the mean 0.5 % slower than the best of the three.  Long launches are held back by the clock that the power
// limit leaves: no faster than the table's PFLOP/s on whole tiles.  128 x 128: 2.9 with batches copied as rows (2.3 before: M = 1894, N = 8448,
// K = 13824 198 us where the sum says 135).  Of 130 drawn calls that 2.3 sent to the whole-tile kernel and 2.9 does not, 126 are faster here, all 1.26
// times in the mean, on row-major weights up to 1.9 times (M = 1355, N = 2688, K = 18944 94.5 -> 49.9 us; tile-major M = 1381, N = 5632,
// K = 7488 44.9 -> 40.9), four slower, many tokens of few feature tiles, which runs along the features (cheapest_order) have made the faster ones
// too (M = 6430, N = 1280, K = 12288 65 -> 77, now 50 as all MXFP4, 73 -> 78 -> 60 on row-major weights).  With 3.3 the
// further ones gain 2 % in the mean.
TilePlanChoice mixed_gemm_tile_plan(int M, int N, int KN, int KS, int KO, int cus) {
  static const struct { int tf, tt; double fixed, round, stage, fill, mb, rest, pflops; } kTiles[] = {
      {128, 128, 2.87, -0.24, 0.260, 0.075, 0.41, 1.8, 2.9}, {128, 64, 1.47, 1.29, 0.170, 0.051, 0.39, 1.0, 2.0}, {64, 64, 1.55, 1.07, 0.125, 0.039, 0.46, 0.9, 1.5}};
  const int stages = KN / 128 + KS / 128 + KO / 128;
  const bool rest = ((KN | KS | KO) & 127) != 0;
  TilePlanChoice best = {0, 0, 0.0};
  for (const auto& t : kTiles) {
    const int64_t tiles = (int64_t)ceil_div(N, t.tf) * ceil_div(M, t.tt);
    const double rounds = (double)((tiles + cus - 1) / cus), busy = tiles < cus ? (double)tiles / cus : 1.0;
    const double power = 2e-9 * (double)tiles * t.tf * t.tt * (KN + KS + KO) / t.pflops;
    const double us = fmax(power, t.fixed + rounds * (t.round + stages * t.stage + (rest ? t.rest : 0.0)) + stages * t.fill * busy + 2e-6 * M * N * t.mb);
    if (best.tf == 0 || us < best.us) best = {t.tf, t.tt, us};
  }
  return best;
}

hipError_t launch_mixed_gemm_tile(const uint8_t* an, const uint8_t* bn, const uint8_t* as_, const uint8_t* bs,
                                  const uint8_t* ao, const uint8_t* bo, const uint8_t* sfan, const uint8_t* sfbn,
                                  const uint8_t* sfas, const uint8_t* sfbs, const uint8_t* sfao, const uint8_t* sfbo,
                                  int m_store, int a_rows, int a_staged, int N, int KN, int KS, int KO, bool w_tiled, const TilePlanChoice& choice,
                                  Epilogue ep, void* d, hipStream_t stream) {
  const int tf = choice.tf, tt = choice.tt;
  if (m_store <= 0 || a_rows < m_store || (a_staged != 0 && (a_staged < a_rows || !staged_in_reach(a_staged)))) return hipErrorInvalidValue;
  TilePlan p;
  p.s4 = {an, bn, sfan, sfbn, KN / 32, KN / 128};
  p.s6 = {as_, bs, sfas, sfbs, KS / 32, KS / 128};
  p.s8 = {ao, bo, sfao, sfbo, KO / 32, KO / 128};
  p.total = p.s4.whole + p.s6.whole + p.s8.whole;
  p.N = N;
  p.m_store = m_store;
  p.a_rows = a_rows;
  p.a_staged = a_staged;
  p.order = cheapest_order(ceil_div(ep.n_out, tf), ceil_div(m_store, tt), tf, tt);
  const bool rem = ((KN | KS | KO) & 127) != 0;
  uint16_t* out = static_cast<uint16_t*>(d);
  if (tf == 128 && tt == 128) return launch_geo<128, 128, 2, 2>(p, w_tiled, rem, ep, out, stream);
  if (tf == 128 && tt == 64) return launch_geo<128, 64, 2, 2>(p, w_tiled, rem, ep, out, stream);
  if (tf == 64 && tt == 64) return launch_geo<64, 64, 1, 4>(p, w_tiled, rem, ep, out, stream);
  return hipErrorInvalidValue;
}

}  // namespace mg
