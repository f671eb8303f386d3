// Products over permuted bf16 rows, see kmoe_gemm_tile.h.
#include "kmoe_gemm_tile.h"

namespace kmoe_tiles {
void launch_permuted(const GemmLaunch& l, bool gate_up) {
  if (gate_up)
    launch_variant<true, false, false>(l);
  else
    launch_variant<false, false, false>(l);
}
}  // namespace kmoe_tiles
