// Host program of tests/test_tile_order_cpu.py: maps every workgroup of each grid given as "tiles_n tiles_m tf tt" on stdin to its
// tile and prints the grids where some tile is not computed exactly once.
#include <stdio.h>

#include <vector>

#include "../../mixedgemm_amd/csrc/tile_order.h"

int main() {
  int tiles_n, tiles_m, tf, tt, grids = 0;
  while (scanf("%d %d %d %d", &tiles_n, &tiles_m, &tf, &tt) == 4) {
    const mg::TileOrder order = mg::tile_order(tiles_n, tiles_m, tf, tt);
    const int nwg = tiles_n * tiles_m;
    std::vector<bool> seen(nwg, false);
    const int rows = mg::grid_rows(order);
    if (order.grid_x > mg::kMostTilesAcross || (long long)order.grid_x * rows < nwg || (long long)order.grid_x * (rows - 1) >= nwg)
      printf("%d x %d tiles of %d x %d: a grid of %d x %d\n", tiles_n, tiles_m, tf, tt, order.grid_x, rows);
    for (int wg = 0; wg < nwg; ++wg) {
      int tn = -1, tm = -1;
      mg::tile_at(order, wg, tn, tm);
      if (tn < 0 || tn >= tiles_n || tm < 0 || tm >= tiles_m || seen[(size_t)tn * tiles_m + tm]) {
        printf("%d x %d tiles of %d x %d: workgroup %d -> (%d, %d)\n", tiles_n, tiles_m, tf, tt, wg, tn, tm);
        break;
      }
      seen[(size_t)tn * tiles_m + tm] = true;
    }
    // where the counts do not divide into rectangles, an XCD's tiles are a run in feature-major order
    for (int xcd = 0; xcd < 8 && (nwg & 7) != 0; ++xcd) {
      int tn, tm, next = -1;
      for (int wg = xcd; wg < nwg; wg += 8) {
        mg::tile_at(order, wg, tn, tm);
        if (next >= 0 && tn * tiles_m + tm != next) {
          printf("%d x %d tiles of %d x %d: no run on XCD %d at workgroup %d\n", tiles_n, tiles_m, tf, tt, xcd, wg);
          break;
        }
        next = tn * tiles_m + tm + 1;
      }
    }
    // runs whatever the counts (the skinny kernel's): every tile once, consecutive on an XCD
    const mg::TileOrder runs = mg::tile_runs(tiles_n, tiles_m);
    std::vector<bool> ran(nwg, false);
    for (int xcd = 0; xcd < 8; ++xcd) {
      int next = -1;
      for (int wg = xcd; wg < nwg; wg += 8) {
        int tn = -1, tm = -1;
        mg::tile_at(runs, wg, tn, tm);
        const bool inside = tn >= 0 && tn < tiles_n && tm >= 0 && tm < tiles_m;
        if (!inside || ran[(size_t)tn * tiles_m + tm] || (next >= 0 && tn * tiles_m + tm != next)) {
          printf("%d x %d tiles in runs: workgroup %d -> (%d, %d)\n", tiles_n, tiles_m, wg, tn, tm);
          break;
        }
        ran[(size_t)tn * tiles_m + tm] = true;
        next = tn * tiles_m + tm + 1;
      }
    }
    ++grids;
  }
  printf("%d grids\n", grids);
  return 0;
}
