// Host program of tests/test_staged_codes_cpu.py: for each "kernel w_tiled rows" on stdin, the rows whose codes go stage by stage.
#include <stdio.h>

#include "../../mixedgemm_amd/csrc/staged_codes.h"

int main() {
  int kernel, w_tiled, rows;
  while (scanf("%d %d %d", &kernel, &w_tiled, &rows) == 3) printf("%d\n", mg::staged_rows(kernel, w_tiled != 0, rows));
  return 0;
}
