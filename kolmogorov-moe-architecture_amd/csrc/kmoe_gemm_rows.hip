// Gathered gate/up products (inference), see kmoe_gemm_tile.h.
#include "kmoe_gemm_tile.h"

namespace kmoe_tiles {
void launch_gate_up_rows(const GemmLaunch& l) {
  if (l.g.a_scale)
    launch_variant<true, false, true, false, true>(l);
  else
    launch_variant<true, false, true>(l);
}
}  // namespace kmoe_tiles
