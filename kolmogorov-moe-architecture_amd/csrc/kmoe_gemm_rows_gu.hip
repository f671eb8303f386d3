// Gathered gate/up product of the training forward, see kmoe_gemm_tile.h.
#include "kmoe_gemm_tile.h"

namespace kmoe_tiles {
void launch_gate_up_rows_gu(const GemmLaunch& l) { launch_variant<true, false, true, true>(l); }
}  // namespace kmoe_tiles
