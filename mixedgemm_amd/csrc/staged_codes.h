// Which layer calls hand their GEMM the codes of the tokens stage by stage (see launch_reorder_quant): a rule for the host.
#pragma once
#include <stdint.h>

#include "../../include/mixedgemm_abi.h"

namespace mg {

// Whether such codes of `rows` rows of up to 128 bytes are in reach of the GEMMs on tiles: they step from one stage to the next by 32 bits (as
// 64 bits the steps have 4 to 13 more scalar registers spilled in the kernel on whole tiles).  2^25 rows and more stay row-major, where a step
// is the 64 ... 128 bytes of one row.
inline bool staged_in_reach(int rows) { return (uint64_t)rows * 128 < (uint64_t)1 << 32; }

// Rows of the workspace (`padded`) for a call whose GEMM is `kernel` (MG_KERNEL_*) if its codes go stage by stage, 0 if row by row.  Whole tiles,
// and small ones on tile-major weights, read whole lines that way; on row-major weights small tiles copy batches of rows, weights and tokens alike.
inline int staged_rows(int kernel, bool w_tiled, int padded) {
  const bool wanted = kernel == MG_KERNEL_WHOLE || (kernel == MG_KERNEL_TILE && w_tiled);
  return wanted && staged_in_reach(padded) ? padded : 0;
}

}  // namespace mg
