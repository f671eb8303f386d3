// Products over e4m3 rows, see kmoe_gemm_tile.h.
#include "kmoe_gemm_tile.h"

namespace kmoe_tiles {
void launch_fp8(const GemmLaunch& l, bool gate_up, bool save_gu) {
  if (save_gu)
    launch_variant<true, true, false, true>(l);
  else if (gate_up)
    launch_variant<true, true, false>(l);
  else
    launch_variant<false, true, false>(l);
}
}  // namespace kmoe_tiles
