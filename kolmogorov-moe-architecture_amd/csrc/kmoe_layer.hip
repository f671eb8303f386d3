// The token-choice layer forward (no gradients) as one call: router, dispatch, expert
// products and combine launched from here, their intermediates in one workspace.  The
// launches are those of the single entry points, in the same order on the same stream.
// From Python the five calls, their argument conversions and some fifteen allocations took
// about 90 us a pass, more than the kernels of a decode step (45 us at one token).
#include "kmoe_common.h"

namespace {

// Buffers of one call in the workspace, 256-byte aligned.
struct Buffers {
  size_t logits, idx, w, partials, hist, offsets, row_token, slot_row, slot_w, dispatch, rscale, h, yperm, total;
};
Buffers layout(int64_t T, int d, int E, int k, int F) {
  Buffers b{};
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t p = at;
    at += (bytes + 255) / 256 * 256;
    return p;
  };
  const size_t A = (size_t)T * k;
  b.logits = take((size_t)T * E * 4);
  b.idx = take(A * 8);
  b.w = take(A * 4);
  b.partials = take((size_t)kmoe_router_partials_len(T, E) * 4);
  b.hist = take((size_t)kmoe::ceil_div<int64_t>(T, kmoe::router_block_tokens(T)) * E * 4);
  b.offsets = take((size_t)(E + 1) * 4);
  b.row_token = take(A * 4);
  b.slot_row = take(A * 4);
  b.slot_w = take(A * 4);
  b.dispatch = take(kmoe_dispatch_workspace_bytes(T, k, E));
  b.rscale = take((size_t)T * 4);
  b.h = take(A * (size_t)kmoe_padded_ff(F) * 2);
  b.yperm = take(A * (size_t)d * 2);
  b.total = at;
  return b;
}

bool valid(int64_t T, int d, int E, int k, int F) {
  return T > 0 && T <= (int64_t)1 << 31 && d > 0 && E >= 1 && E <= KMOE_MAX_EXPERTS && k >= 1 && k <= 8 && F > 0;
}

}  // namespace

extern "C" size_t kmoe_moe_forward_workspace_bytes(int64_t T, int d, int E, int k, int F) {
  return valid(T, d, E, k, F) ? layout(T, d, E, k, F).total : 0;
}

extern "C" int kmoe_moe_forward(const void* x, int64_t T, int d, const void* w_in, const void* w_out, int E,
                                const float* logit_bias, int k, const void* w13_packed, const void* w3_packed, int F,
                                int64_t capacity, float rms_eps, const void* residual, void* y, int y_dtype,
                                int32_t* counts, float* aux_out, float w_lb, float w_z, void* workspace,
                                size_t workspace_bytes, void* stream) {
  KMOE_REQUIRE(x && w_in && w_out && w13_packed && w3_packed && y && counts && workspace, KMOE_ERR_NULL,
               "kmoe_moe_forward: null buffer");
  KMOE_REQUIRE(valid(T, d, E, k, F), KMOE_ERR_SHAPE, "kmoe_moe_forward: T=%lld d=%d E=%d k=%d F=%d", (long long)T, d,
               E, k, F);
  const Buffers b = layout(T, d, E, k, F);
  KMOE_REQUIRE(workspace_bytes >= b.total, KMOE_ERR_WORKSPACE, "kmoe_moe_forward: workspace %zu < %zu bytes",
               workspace_bytes, b.total);
  uint8_t* const ws = static_cast<uint8_t*>(workspace);
  auto f32 = [&](size_t at) { return reinterpret_cast<float*>(ws + at); };
  auto i32 = [&](size_t at) { return reinterpret_cast<int32_t*>(ws + at); };
  int64_t* const idx = reinterpret_cast<int64_t*>(ws + b.idx);
  const bool rms = rms_eps >= 0.0f;
  float* const rscale = rms ? f32(b.rscale) : nullptr;
  int rc = kmoe::router_launch(x, nullptr, T, d, w_in, w_out, E, logit_bias, k, f32(b.logits), idx, f32(b.w),
                               f32(b.partials), nullptr, rms ? rms_eps : 0.0f, rscale, i32(b.hist), stream);
  if (rc) return rc;
  const size_t dws = kmoe_dispatch_workspace_bytes(T, k, E);
  if (aux_out)
    rc = kmoe_dispatch_counted_aux(x, nullptr, T, d, idx, f32(b.w), KMOE_DTYPE_F32, k, E, capacity, i32(b.hist), counts,
                                   i32(b.offsets), i32(b.row_token), i32(b.slot_row), f32(b.slot_w), nullptr,
                                   KMOE_DTYPE_BF16, nullptr, ws + b.dispatch, dws, f32(b.partials), w_lb, w_z, aux_out,
                                   stream);
  else
    rc = kmoe_dispatch_counted(x, nullptr, T, d, idx, f32(b.w), KMOE_DTYPE_F32, k, E, capacity, i32(b.hist), counts,
                               i32(b.offsets), i32(b.row_token), i32(b.slot_row), f32(b.slot_w), nullptr,
                               KMOE_DTYPE_BF16, nullptr, ws + b.dispatch, dws, stream);
  if (rc) return rc;
  const int64_t A = T * k;
  if (rms)
    rc = kmoe_gemm_gate_up_rows_scaled(x, nullptr, T, i32(b.row_token), i32(b.offsets), E, d, F, A, w13_packed, rscale,
                                       ws + b.h, stream);
  else
    rc = kmoe_gemm_gate_up_rows(x, nullptr, T, i32(b.row_token), i32(b.offsets), E, d, F, A, w13_packed, ws + b.h,
                                stream);
  if (rc) return rc;
  rc = kmoe_gemm_down(ws + b.h, nullptr, KMOE_DTYPE_BF16, i32(b.offsets), E, d, F, A, w3_packed, nullptr, ws + b.yperm,
                      stream);
  if (rc) return rc;
  return kmoe_combine_residual(ws + b.yperm, d, i32(b.slot_row), f32(b.slot_w), k, nullptr, nullptr, residual, T, y,
                               y_dtype, stream);
}
