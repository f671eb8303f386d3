// Grouped expert products: launch choice and C entry points.  The kernels are in
// kmoe_gemm_tile.h.
#include <algorithm>

#include "kmoe_gemm_tile.h"

using namespace kmoe_tiles;

namespace {

// Slots of SMALL_ROWS rows that max_rows rows over E experts can fill: at most one per row,
// and the full ones plus a partial one per expert.
int64_t small_slots(int E, int64_t max_rows) { return std::min<int64_t>(max_rows, max_rows / SMALL_ROWS + E); }

// Whether a bf16 product runs on the small-row kernel and not on the 256-row tiles.  Kernel
// times in us, small-row kernel / 256-row tiles, weights not in a cache, top-2:
// - where its grid is at most two workgroups per CU, as latency then counts: d 256, F 352, 4
//   experts: 128 tokens 10.0 / 15.9, 512 tokens 15.9 / 16.3 (down 6.3 / 8.2 at 288
//   workgroups, gate/up 9.6 / 8.2 at 864);
// - and at few rows per expert (max_rows / E), where the weights are the traffic and are read
//   once: up to 6 where one tile per expert and column tile fills the CUs in whole rounds or
//   in more than two, else up to 10.  Gate/up and down at 4, 8 and 10 rows each: 64 experts, d
//   2048, F 1408 (704 and 512 tiles) 125 / 134 and 65 / 69, 134 / 135 and 69 / 69, 140 / 135
//   and 71 / 70; 32 experts, d 2048, F 768 (192 and 256) 38.6 / 41.3 and 25.5 / 23.2, 38.7 /
//   39.4 and 25.6 / 22.8; 16 experts, d 2048, F 2816 (352 and 128) 66 / 81 and 36 / 43, 70 / 81
//   and 38 / 43, 72 / 81 and 40 / 43; 8 experts, d 2048, F 2816 (176 and 64) 37 / 40 and 20 /
//   33, 38 / 39 and 21 / 33, 39 / 37 and 20 / 32.  At 16 rows: 159 / 136 and 81 / 70 (64
//   experts), 79 / 77 and 42 / 40 (16), 43 / 38 and 22 / 32 (8);
// - if not too many workgroups stream one expert's weights again for its further slots: at
//   most three per CU over the full slots that the rows can make.  All rows on one expert,
//   gate/up and down: 16 experts, 64 rows (352 workgroups in gate/up) 18 / 21 and 13 / 26, 128
//   rows (704) 26 / 21 and 13 / 26, 160 rows (880) 33 / 21 and 23 / 26; 64 experts, 256 rows
//   (704) 26 / 21 and 15 / 15, 640 rows (1760) 56 / 22 and 31 / 16.  (Zipf 1.2 routing: 0.75
//   to 1.08 of the tiles' time in gate/up, 0.7 to 1.06 in down.)
// (A kernel of 128-row slots for 10 to 64 rows per expert, weights to registers and rows
// through LDS, measured 4% faster alone at 16 to 32 rows and 2% slower inside a layer.)
bool small_rows_product(bool gate_up, int E, int64_t max_rows, int64_t b_expert_rows, int64_t ldb_bytes,
                        int n_tiles) {
  // lanes address an expert's weights with 31-bit offsets
  if (b_expert_rows * ldb_bytes >= (int64_t)1 << 31) return false;
  const int64_t n_ct = (int64_t)n_tiles * (gate_up ? BN / 2 : BN) / small_cols(gate_up);
  const int64_t n_cu = kmoe::cu_count();
  if (small_slots(E, max_rows) * n_ct <= 2 * n_cu) return true;
  const int64_t tiles = (int64_t)E * n_tiles;
  const int rows = tiles % n_cu == 0 || tiles > 2 * n_cu ? 6 : 10;
  // (a launch takes 2^24 workgroups of 256)
  return max_rows <= rows * (int64_t)E && max_rows / SMALL_ROWS * n_ct <= 3 * n_cu &&
         small_slots(E, max_rows) * n_ct < 1 << 24;
}

// A rows: the permuted rows (row_token == nullptr) or gathered rows of the
// activation matrix A (n_a_rows rows) through row_token / row_index.
int launch_gemm(bool gate_up, bool fp8, const void* A, const float* a_scale, const int32_t* row_token,
                const int32_t* row_index, int64_t n_a_rows, const int32_t* offsets, int E, int K, int64_t max_rows,
                const void* B, int64_t b_expert_rows, const float* b_scale, void* C, int64_t ldc, int n_valid,
                int n_tiles, hipStream_t s, void* gu_out = nullptr, int64_t ldb_bytes = 0, const void* B2 = nullptr) {
  const int eb = fp8 ? 1 : 2;
  const int64_t slots = kmoe::ceil_div<int64_t>(max_rows, BM) + E;
  const int n_cu = kmoe::cu_count();
  const int kbytes = K * eb;
  if (kbytes % KB != 0) {
    kmoe::set_error("kmoe gemm: K bytes %d not a multiple of %d", kbytes, KB);
    return KMOE_ERR_SHAPE;
  }
  GemmArgs g{};  // value-initialised: every optional output starts null
  g.A = static_cast<const uint8_t*>(A);
  g.lda_bytes = kbytes;
  g.a_scale = a_scale;
  g.row_token = row_token;
  g.row_index = row_index;
  g.B = static_cast<const uint8_t*>(B);
  g.b_expert_rows = b_expert_rows;
  g.B2 = static_cast<const uint8_t*>(B2);
  g.ldb_bytes = ldb_bytes ? ldb_bytes : kbytes + WPAD;
  g.b_scale = b_scale;
  g.k_bytes = kbytes;
  g.C = static_cast<uint16_t*>(C);
  g.ldc = ldc;
  g.n_valid = n_valid;
  g.gu_out = static_cast<uint16_t*>(gu_out);
  // every tile of the worst-case slot count, plus one narrow tile per resident
  // workgroup for the split tail
  int64_t blocks = slots * n_tiles + n_cu;
  if (blocks > 0x7fffffff) {
    kmoe::set_error("kmoe gemm: grid too large");
    return KMOE_ERR_SHAPE;
  }
  // e4m3: one workgroup per CU for the full-tile loop and one for the narrow tiles after it;
  // without the loop every tile in halves, or in quarters on at most n_cu workgroups
  if (fp8) blocks = full_tile_loop(g) ? 2 * n_cu : std::max<int64_t>(2 * slots * n_tiles, n_cu);
  // tile loads address a 2 GiB buffer window from the tile's first A / B row (from
  // the first row of A when gathering); with B2 a row of A is twice one of B
  if ((int64_t)(BM + 1) * std::max(g.lda_bytes, g.ldb_bytes) >= ((int64_t)1 << 31) ||
      (row_token && (n_a_rows + 1) * g.lda_bytes >= ((int64_t)1 << 31))) {
    kmoe::set_error("kmoe gemm: operand too large for 32-bit tile offsets (K bytes %d)", kbytes);
    return KMOE_ERR_SHAPE;
  }
  const GemmLaunch l{g, offsets, E, n_tiles, n_cu, (unsigned)blocks, s};
  if (!fp8 && small_rows_product(gate_up, E, max_rows, b_expert_rows, g.ldb_bytes, n_tiles)) {
    const int n_ct = n_tiles * (gate_up ? BN / 2 : BN) / small_cols(gate_up);
    launch_small_rows(GemmLaunch{g, offsets, E, n_ct, n_cu, (unsigned)(small_slots(E, max_rows) * n_ct), s}, gate_up);
  } else if (B2)
    launch_dual(l);
  else if (fp8)
    launch_fp8(l, gate_up, gu_out != nullptr);
  else if (row_token && gu_out)
    launch_gate_up_rows_gu(l);
  else if (row_token)
    launch_gate_up_rows(l);
  else
    launch_permuted(l, gate_up);
  return KMOE_OK;
}

}  // namespace

static int check_gemm_args(const char* who, const void* a, const int32_t* offsets, int E, int d, int F,
                           int64_t max_rows, const void* w, const void* out, int in_dtype) {
  KMOE_REQUIRE(a && offsets && w && out, KMOE_ERR_NULL, "%s: null buffer", who);
  KMOE_REQUIRE(E >= 1 && E <= KMOE_MAX_EXPERTS, KMOE_ERR_SHAPE, "%s: E=%d out of range", who, E);
  KMOE_REQUIRE(d > 0 && d % 64 == 0, KMOE_ERR_SHAPE, "%s: d=%d must be a positive multiple of 64", who, d);
  KMOE_REQUIRE(F > 0, KMOE_ERR_SHAPE, "%s: F=%d must be > 0", who, F);
  KMOE_REQUIRE(max_rows >= 0 && max_rows < ((int64_t)1 << 31), KMOE_ERR_SHAPE, "%s: max_rows out of range", who);
  KMOE_REQUIRE(in_dtype == KMOE_DTYPE_BF16 || in_dtype == KMOE_DTYPE_FP8_E4M3, KMOE_ERR_DTYPE,
               "%s: input dtype must be bf16 or fp8_e4m3", who);
  return KMOE_OK;
}

extern "C" int kmoe_gemm_gate_up(const void* xperm, const float* xperm_scale, int in_dtype, const int32_t* offsets,
                                 int E, int d, int F, int64_t max_rows, const void* w13_packed, const float* w13_scale,
                                 void* h, void* stream) {
  int rc = check_gemm_args("kmoe_gemm_gate_up", xperm, offsets, E, d, F, max_rows, w13_packed, h, in_dtype);
  if (rc) return rc;
  const bool fp8 = in_dtype == KMOE_DTYPE_FP8_E4M3;
  KMOE_REQUIRE(!fp8 || (xperm_scale && w13_scale), KMOE_ERR_NULL, "kmoe_gemm_gate_up: fp8 needs scales");
  KMOE_REQUIRE(!fp8 || d % 128 == 0, KMOE_ERR_SHAPE, "kmoe_gemm_gate_up: fp8 needs d %% 128 == 0 (d=%d)", d);
  if (max_rows == 0) return KMOE_OK;
  const int Fp = round_up(F, 128);
  rc = launch_gemm(true, fp8, xperm, xperm_scale, nullptr, nullptr, 0, offsets, E, d, max_rows, w13_packed,
                   2 * (int64_t)Fp, w13_scale, h, Fp, Fp, Fp / 128, kmoe::as_stream(stream));
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_gate_up");
}

extern "C" int kmoe_gemm_gate_up_rows(const void* x, const int32_t* row_index, int64_t n_x_rows,
                                      const int32_t* row_token, const int32_t* offsets, int E, int d, int F,
                                      int64_t max_rows, const void* w13_packed, void* h, void* stream) {
  int rc = check_gemm_args("kmoe_gemm_gate_up_rows", x, offsets, E, d, F, max_rows, w13_packed, h, KMOE_DTYPE_BF16);
  if (rc) return rc;
  KMOE_REQUIRE(row_token, KMOE_ERR_NULL, "kmoe_gemm_gate_up_rows: null row_token");
  KMOE_REQUIRE(n_x_rows >= 1, KMOE_ERR_SHAPE, "kmoe_gemm_gate_up_rows: n_x_rows=%lld must be >= 1",
               (long long)n_x_rows);
  if (max_rows == 0) return KMOE_OK;
  const int Fp = round_up(F, 128);
  rc = launch_gemm(true, false, x, nullptr, row_token, row_index, n_x_rows, offsets, E, d, max_rows, w13_packed,
                   2 * (int64_t)Fp, nullptr, h, Fp, Fp, Fp / 128, kmoe::as_stream(stream));
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_gate_up_rows");
}

extern "C" int kmoe_gemm_gate_up_rows_scaled(const void* x, const int32_t* row_index, int64_t n_x_rows,
                                             const int32_t* row_token, const int32_t* offsets, int E, int d, int F,
                                             int64_t max_rows, const void* w13_packed, const float* rscale, void* h,
                                             void* stream) {
  int rc = check_gemm_args("kmoe_gemm_gate_up_rows_scaled", x, offsets, E, d, F, max_rows, w13_packed, h,
                           KMOE_DTYPE_BF16);
  if (rc) return rc;
  KMOE_REQUIRE(row_token && rscale, KMOE_ERR_NULL, "kmoe_gemm_gate_up_rows_scaled: null row_token / rscale");
  KMOE_REQUIRE(n_x_rows >= 1, KMOE_ERR_SHAPE, "kmoe_gemm_gate_up_rows_scaled: n_x_rows=%lld must be >= 1",
               (long long)n_x_rows);
  if (max_rows == 0) return KMOE_OK;
  const int Fp = round_up(F, 128);
  rc = launch_gemm(true, false, x, rscale, row_token, row_index, n_x_rows, offsets, E, d, max_rows, w13_packed,
                   2 * (int64_t)Fp, nullptr, h, Fp, Fp, Fp / 128, kmoe::as_stream(stream));
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_gate_up_rows_scaled");
}

extern "C" int kmoe_gemm_down(const void* h, const float* h_scale, int in_dtype, const int32_t* offsets, int E, int d,
                              int F, int64_t max_rows, const void* w3_packed, const float* w3_scale, void* y,
                              void* stream) {
  int rc = check_gemm_args("kmoe_gemm_down", h, offsets, E, d, F, max_rows, w3_packed, y, in_dtype);
  if (rc) return rc;
  const bool fp8 = in_dtype == KMOE_DTYPE_FP8_E4M3;
  KMOE_REQUIRE(!fp8 || (h_scale && w3_scale), KMOE_ERR_NULL, "kmoe_gemm_down: fp8 needs scales");
  if (max_rows == 0) return KMOE_OK;
  const int Fp = round_up(F, 128), dp = round_up(d, 256);
  rc = launch_gemm(false, fp8, h, h_scale, nullptr, nullptr, 0, offsets, E, Fp, max_rows, w3_packed, dp, w3_scale, y,
                   d, d, dp / BN, kmoe::as_stream(stream));
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_down");
}

extern "C" int kmoe_grouped_swiglu(const void* xperm, const int32_t* offsets, int E, int d, int F, int64_t max_rows,
                                   const void* w13_packed, const void* w3_packed, void* h, void* y, void* stream) {
  int rc = kmoe_gemm_gate_up(xperm, nullptr, KMOE_DTYPE_BF16, offsets, E, d, F, max_rows, w13_packed, nullptr, h,
                             stream);
  if (rc) return rc;
  return kmoe_gemm_down(h, nullptr, KMOE_DTYPE_BF16, offsets, E, d, F, max_rows, w3_packed, nullptr, y, stream);
}

// ---------------------------------------------------------------- backward pass

extern "C" int kmoe_gemm_gate_up_rows_gu(const void* x, const int32_t* row_index, int64_t n_x_rows,
                                         const int32_t* row_token, const int32_t* offsets, int E, int d, int F,
                                         int64_t max_rows, const void* w13_packed, void* h, void* gu, void* stream) {
  int rc = check_gemm_args("kmoe_gemm_gate_up_rows_gu", x, offsets, E, d, F, max_rows, w13_packed, h,
                           KMOE_DTYPE_BF16);
  if (rc) return rc;
  KMOE_REQUIRE(row_token && gu, KMOE_ERR_NULL, "kmoe_gemm_gate_up_rows_gu: null row_token / gu");
  KMOE_REQUIRE(n_x_rows >= 1, KMOE_ERR_SHAPE, "kmoe_gemm_gate_up_rows_gu: n_x_rows=%lld must be >= 1",
               (long long)n_x_rows);
  if (max_rows == 0) return KMOE_OK;
  const int Fp = round_up(F, 128);
  rc = launch_gemm(true, false, x, nullptr, row_token, row_index, n_x_rows, offsets, E, d, max_rows, w13_packed,
                   2 * (int64_t)Fp, nullptr, h, Fp, Fp, Fp / 128, kmoe::as_stream(stream), gu);
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_gate_up_rows_gu");
}

extern "C" int kmoe_gemm_gate_up_fp8_gu(const void* xperm, const float* xperm_scale, const int32_t* offsets, int E,
                                        int d, int F, int64_t max_rows, const void* w13_packed, const float* w13_scale,
                                        void* h, void* gu, void* stream) {
  int rc = check_gemm_args("kmoe_gemm_gate_up_fp8_gu", xperm, offsets, E, d, F, max_rows, w13_packed, h,
                           KMOE_DTYPE_FP8_E4M3);
  if (rc) return rc;
  KMOE_REQUIRE(xperm_scale && w13_scale && gu, KMOE_ERR_NULL, "kmoe_gemm_gate_up_fp8_gu: null scale / gu");
  KMOE_REQUIRE(d % 128 == 0, KMOE_ERR_SHAPE, "kmoe_gemm_gate_up_fp8_gu: fp8 needs d %% 128 == 0 (d=%d)", d);
  if (max_rows == 0) return KMOE_OK;
  const int Fp = round_up(F, 128);
  rc = launch_gemm(true, true, xperm, xperm_scale, nullptr, nullptr, 0, offsets, E, d, max_rows, w13_packed,
                   2 * (int64_t)Fp, w13_scale, h, Fp, Fp, Fp / 128, kmoe::as_stream(stream), gu);
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_gate_up_fp8_gu");
}

extern "C" int kmoe_gemm_grouped(const void* a, const int32_t* offsets, int E, int K, int64_t max_rows,
                                 const void* b_packed, int64_t b_expert_rows, int N, void* c, int64_t ldc, int n_valid,
                                 void* stream) {
  KMOE_REQUIRE(a && offsets && b_packed && c, KMOE_ERR_NULL, "kmoe_gemm_grouped: null buffer");
  KMOE_REQUIRE(E >= 1 && E <= KMOE_MAX_EXPERTS, KMOE_ERR_SHAPE, "kmoe_gemm_grouped: E=%d out of range", E);
  KMOE_REQUIRE(K > 0 && K % 64 == 0, KMOE_ERR_SHAPE, "kmoe_gemm_grouped: K=%d must be a positive multiple of 64", K);
  KMOE_REQUIRE(N > 0 && b_expert_rows >= round_up(N, BN) && b_expert_rows % BN == 0, KMOE_ERR_SHAPE,
               "kmoe_gemm_grouped: b_expert_rows=%lld must be a multiple of %d covering N=%d",
               (long long)b_expert_rows, BN, N);
  KMOE_REQUIRE(n_valid > 0 && n_valid <= ldc, KMOE_ERR_SHAPE, "kmoe_gemm_grouped: n_valid=%d, ldc=%lld", n_valid,
               (long long)ldc);
  KMOE_REQUIRE(max_rows >= 0 && max_rows < ((int64_t)1 << 31), KMOE_ERR_SHAPE, "kmoe_gemm_grouped: max_rows");
  if (max_rows == 0) return KMOE_OK;
  const int rc = launch_gemm(false, false, a, nullptr, nullptr, nullptr, 0, offsets, E, K, max_rows, b_packed,
                             b_expert_rows, nullptr, c, ldc, n_valid, (int)(round_up(N, BN) / BN),
                             kmoe::as_stream(stream));
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_grouped");
}

extern "C" int kmoe_gemm_grouped_weights(const void* a, const int32_t* offsets, int E, int K, int64_t max_rows,
                                         const void* b, const void* b2, int N, void* c, int64_t ldc, void* stream) {
  KMOE_REQUIRE(a && offsets && b && c, KMOE_ERR_NULL, "kmoe_gemm_grouped_weights: null buffer");
  KMOE_REQUIRE(E >= 1 && E <= KMOE_MAX_EXPERTS, KMOE_ERR_SHAPE, "kmoe_gemm_grouped_weights: E=%d out of range", E);
  // whole tiles of weight rows and of columns: nothing past a matrix's end is read
  KMOE_REQUIRE(K > 0 && K % (b2 ? 256 : 64) == 0 && N > 0 && N % BN == 0 && N <= ldc, KMOE_ERR_SHAPE,
               "kmoe_gemm_grouped_weights: K=%d, N=%d, ldc=%lld", K, N, (long long)ldc);
  KMOE_REQUIRE(((reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(b2)) & 15) == 0, KMOE_ERR_SHAPE,
               "kmoe_gemm_grouped_weights: weights not aligned to 16 bytes");
  KMOE_REQUIRE(max_rows >= 0 && max_rows < ((int64_t)1 << 31), KMOE_ERR_SHAPE, "kmoe_gemm_grouped_weights: max_rows");
  if (max_rows == 0) return KMOE_OK;
  const int rc = launch_gemm(false, false, a, nullptr, nullptr, nullptr, 0, offsets, E, K, max_rows, b, N, nullptr, c,
                             ldc, N, N / BN, kmoe::as_stream(stream), nullptr, (int64_t)K * (b2 ? 1 : 2), b2);
  if (rc) return rc;
  return kmoe::check_launch("kmoe_gemm_grouped_weights");
}
