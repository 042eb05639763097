// Which tile of the result a workgroup of the small-tile GEMM computes: integer arithmetic for the kernel and for the host.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mg {

// Workgroups go to the 8 XCDs round-robin; an XCD (an L2) gets a rectangle of tiles where the counts divide, the one with the fewest
// operand bytes per stage, else a run of consecutive tiles in feature-major order (the runs of the first XCDs one tile longer).
// (Dealt out one by one where the number of tiles is no multiple of 8, all XCDs fetched all weights, once per tile of tokens: M = 140,
// N = 18944, K = 8192 from the last-level cache 40.9 us, now 31.3; M = 263, N = 17152, K = 13824 96.6, now 65.3; 359 such calls
// 1.09 times as fast in the mean, 235 from HBM 1.03.)
struct TileOrder {
  // A rectangle of `div` x div2 tiles per XCD, 2^xlog rectangles along the features, or (xlog < 0) runs of at least div2 tiles: token tile
  // after token tile (-1; div = token tiles) or feature tile after feature tile (-2; div = feature tiles)
  int xlog, div, div2;
  unsigned magic;   // 2^32 / div, rounded up (div > 1)
  int grid_x, tiles;   // workgroups per row of the launch grid, and of all
};

// HIP takes fewer than 2^32 threads along a dimension of a grid; a launch of more tiles than this has several rows of workgroups.
constexpr int kMostTilesAcross = 1 << 22;   // of at most 1023 threads each

// Runs of consecutive tiles, token tile after token tile, whatever the counts.
inline TileOrder tile_runs(int tiles_n, int tiles_m) {
  const int nwg = tiles_n * tiles_m;
  return {-1, tiles_m, nwg >> 3, tiles_m > 1 ? (unsigned)(((1ull << 32) + tiles_m - 1) / tiles_m) : 0,
          nwg < kMostTilesAcross ? nwg : kMostTilesAcross, nwg};
}

// tf x tt: features and tokens of a tile
inline TileOrder tile_order(int tiles_n, int tiles_m, int tf, int tt) {
  TileOrder o = tile_runs(tiles_n, tiles_m);
  const int nwg = o.tiles;
  if ((nwg & 7) == 0) {
    double best = 0.0;
    for (int x = 3; x >= 0; --x) {
      const int gx = 1 << x, gy = 8 >> x;
      if (tiles_n % gx || tiles_m % gy) continue;
      const double cost = (double)(tiles_n / gx) * tf * 64 + (double)(tiles_m / gy) * tt * 80;   // operand bytes per stage of a rectangle
      if (o.xlog < 0 || cost < best) {
        best = cost;
        o.xlog = x;
        o.div = tiles_n / gx;
        o.div2 = tiles_m / gy;
      }
    }
  }
  o.magic = o.div > 1 ? (unsigned)(((1ull << 32) + o.div - 1) / o.div) : 0;
  return o;
}

// What the small-tile GEMM is launched with: tile_order, but runs along the features where those of an XCD are four fifths of the operand bytes per stage or less (many
// tokens of few features: 51 x 10 tiles in runs along the tokens had every L2 fetch nearly all tokens).  GEMM alone, us: M = 6430, N = 1280, K = 12288 66.0 -> 50.5
// (tile-major), 78.0 -> 60.2 (row-major); M = 3694, N = 896, K = 7872 26.8 -> 21.0; M = 2874, N = 1152, K = 4096 12.6 -> 10.8; M = 1339, N = 640, K = 1792 6.3 -> 5.4; of
// 76 calls of 256 ... 6500 tokens 26 have such runs and gain 7 % in the mean, the others are as before.  Only where they are a fifth fewer: 14 calls with 2 ... 19 %
// fewer are level either way (at most 3 %, 0.5 % in the mean, as much as two runs of one side).
inline TileOrder cheapest_order(int tiles_n, int tiles_m, int tf, int tt) {
  TileOrder o = tile_order(tiles_n, tiles_m, tf, tt);
  if (o.xlog >= 0) return o;
  // bytes of the tiles that a run of `length` touches: across whole lines of `line` tiles, and along one
  const int length = (o.tiles >> 3) + 1;
  auto touched = [&](int line, int lines, int of_line, int across) {
    const int n = (length + line - 2) / line + 1;
    return (double)(n < lines ? n : lines) * across + (double)(length < line ? length : line) * of_line;
  };
  if (touched(tiles_n, tiles_m, tf * 64, tt * 80) < 0.8 * touched(tiles_m, tiles_n, tt * 80, tf * 64)) {
    o.xlog = -2;
    o.div = tiles_n;
    o.magic = o.div > 1 ? (unsigned)(((1ull << 32) + o.div - 1) / o.div) : 0;
  }
  return o;
}

inline int grid_rows(const TileOrder& o) { return (int)(((int64_t)o.tiles + o.grid_x - 1) / o.grid_x); }

// wg: the workgroup's number in launch order, below o.tiles
__host__ __device__ inline void tile_at(const TileOrder& o, int wg, int& tn, int& tm) {
  const int xcd = wg & 7;
  int j = wg >> 3;
  if (o.xlog < 0) j += xcd * o.div2 + (xcd < (o.tiles & 7) ? xcd : o.tiles & 7);
  int q = j, r = 0;
  if (o.div > 1) {
    // magic * div = 2^32 + e with 0 <= e < div, so the product is j / div + (j * e / div) / 2^32: less than one too large for any
    // 31-bit j, and its whole part is j / div or, for some of the j that lie just below a multiple of div, one more.
    q = (int)(((uint64_t)(uint32_t)j * o.magic) >> 32);
    r = j - q * o.div;
    if (r < 0) {
      q -= 1;
      r += o.div;
    }
  }
  if (o.xlog == -1) {
    tn = q;
    tm = r;
  } else if (o.xlog < 0) {
    tn = r;
    tm = q;
  } else {
    tn = (xcd & ((1 << o.xlog) - 1)) * o.div + r;
    tm = (xcd >> o.xlog) * o.div2 + q;
  }
}

}  // namespace mg
