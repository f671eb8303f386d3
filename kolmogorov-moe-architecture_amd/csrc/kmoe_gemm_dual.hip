// Product over permuted bf16 rows with the weights read from two matrices, see dual_step_second
// in kmoe_gemm_tile.h.  The rows have no padding behind them (d 2048: 4 KiB apart, w1 and w2
// of F 2816: 5.5 KiB); 4096 tokens, top-2 of 16 experts: dx 168 us, dh + dx 363 us against
// 365 us of the packed copies, whose making took 207 us.
#include "kmoe_gemm_tile.h"

namespace kmoe_tiles {
void launch_dual(const GemmLaunch& l) { launch_variant<false, false, false, false, false, true>(l); }
}  // namespace kmoe_tiles
