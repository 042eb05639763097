// Host program of tests/test_tile_order_cpu.py: every tile of each grid given as "tiles_n tiles_m tf tt" on stdin is computed exactly once in
// the order that the small-tile GEMM is launched with; prints the grids where it is not, and how many have runs along the features.
#include <stdio.h>

#include <vector>

#include "../../mixedgemm_amd/csrc/tile_order.h"

int main() {
  int tiles_n, tiles_m, tf, tt, columns = 0;
  while (scanf("%d %d %d %d", &tiles_n, &tiles_m, &tf, &tt) == 4) {
    const mg::TileOrder order = mg::cheapest_order(tiles_n, tiles_m, tf, tt);
    const int nwg = tiles_n * tiles_m;
    std::vector<bool> seen(nwg, false);
    for (int xcd = 0; xcd < 8; ++xcd) {
      int next = -1;
      for (int wg = xcd; wg < nwg; wg += 8) {
        int tn = -1, tm = -1;
        mg::tile_at(order, wg, tn, tm);
        const bool inside = tn >= 0 && tn < tiles_n && tm >= 0 && tm < tiles_m;
        if (!inside || seen[(size_t)tn * tiles_m + tm] || (order.xlog == -2 && next >= 0 && tm * tiles_n + tn != next)) {
          printf("%d x %d tiles of %d x %d: workgroup %d -> (%d, %d)\n", tiles_n, tiles_m, tf, tt, wg, tn, tm);
          break;
        }
        seen[(size_t)tn * tiles_m + tm] = true;
        next = tm * tiles_n + tn + 1;
      }
    }
    columns += order.xlog == -2;
  }
  printf("%d along the features\n", columns);
  return 0;
}
