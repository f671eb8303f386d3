// Packed layouts of the expert weights (kmoe_gemm_tile.h has the forward's) and per-row fp8
// quantisation.
#include "kmoe_gemm_tile.h"

using namespace kmoe_tiles;

namespace {

// ---------------------------------------------------------------- weight packing
// out[e][map(c)][r] = in[e][r][c] for in (E, R, Cn) row-major; rows of `out` have
// length out_ld (>= R, zero padded), out has out_rows rows per expert (zero padded).
// gate_up maps input column f of w1 (half 0) / w2 (half 1) to packed row
// (f/128)*256 + half*128 + f%128; down maps column n of w3 to row n.
template <bool IN_F32, bool FP8>
__global__ __launch_bounds__(256) void pack_transpose_kernel(const void* __restrict__ in, int R, int Cn,
                                                             int64_t in_expert_stride, int half, bool gate_up,
                                                             uint8_t* __restrict__ out, int64_t out_rows, int out_ld,
                                                             const float* __restrict__ row_scale) {
  __shared__ float tile[64][65];
  const int e = blockIdx.z;
  const int r0 = blockIdx.y * 64;  // input rows (become output columns)
  const int c0 = blockIdx.x * 64;  // input cols (become output rows)
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += 4) {
    const int r = r0 + i, c = c0 + tx;
    float v = 0.0f;
    if (r < R && c < Cn) {
      const int64_t off = (int64_t)e * in_expert_stride + (int64_t)r * Cn + c;
      v = IN_F32 ? static_cast<const float*>(in)[off] : bf16_to_f32(static_cast<const uint16_t*>(in)[off]);
    }
    tile[i][tx] = v;
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    const int c = c0 + i;  // output row source column
    const int r = r0 + tx;  // output column
    if (c >= Cn || r >= out_ld) continue;
    const int64_t orow = gate_up ? (int64_t)(c / 128) * 256 + half * 128 + (c % 128) : (int64_t)c;
    const int64_t o = ((int64_t)e * out_rows + orow) * out_ld + r;
    const float v = tile[tx][i];
    if (FP8) {
      // row_scale holds the row amax at this point (finalised to amax/448 afterwards)
      const float amax = row_scale[(int64_t)e * out_rows + orow];
      const float inv = amax > 0.0f ? 448.0f / amax : 0.0f;
      out[o] = (uint8_t)f32_to_e4m3(v * inv);
    } else {
      reinterpret_cast<uint16_t*>(out)[o] = f32_to_bf16(v);
    }
  }
}

// Column amax of in[e] (R x Cn) -> per packed row amax (turned into amax/448 by
// finalize_scale_kernel once the rows have been quantised).  Workgroup (column block,
// row block, expert): each thread takes the max over COLS_ROWS rows of its column and
// merges it with an integer atomicMax on the float's bits (non-negative floats order
// like their bit patterns; max is order-independent, so the result is deterministic).
// The scale buffer starts at 0 (zero_f32_kernel).
constexpr int COLS_ROWS = 64;
template <bool IN_F32>
__global__ __launch_bounds__(256) void col_scale_kernel(const void* __restrict__ in, int R, int Cn,
                                                        int64_t in_expert_stride, int half, bool gate_up,
                                                        float* __restrict__ scale, int64_t out_rows) {
  const int e = blockIdx.z;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= Cn) return;
  const int r0 = blockIdx.y * COLS_ROWS, r1 = min(R, r0 + COLS_ROWS);
  float amax = 0.0f;
  for (int r = r0; r < r1; ++r) {
    const int64_t off = (int64_t)e * in_expert_stride + (int64_t)r * Cn + c;
    const float v = IN_F32 ? static_cast<const float*>(in)[off] : bf16_to_f32(static_cast<const uint16_t*>(in)[off]);
    amax = fmaxf(amax, fabsf(v));
  }
  const int64_t orow = gate_up ? (int64_t)(c / 128) * 256 + half * 128 + (c % 128) : (int64_t)c;
  atomicMax(reinterpret_cast<unsigned int*>(scale + (int64_t)e * out_rows + orow), __float_as_uint(amax));
}

__global__ void finalize_scale_kernel(float* __restrict__ p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = p[i] / 448.0f;
}

__global__ void zero_kernel(uint8_t* __restrict__ p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}
__global__ void zero_f32_kernel(float* __restrict__ p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0.0f;
}

// bf16 pack of one weight matrix per expert, in[e] (R x Cn) row-major -> out rows
// (out[e][map(c)][r] = in[e][r][c], map as in pack_transpose_kernel), 16 bytes per
// global access: a 64 x 64 tile is read as 8-element row vectors (bf16 16 B, f32 2 x
// 16 B), transposed through LDS, and written as 8-element vectors of output rows.
// Entries of out that no input element maps to (the pad after each row, padding
// rows) are left alone (pack_pad_kernel zeroes them).
template <bool IN_F32>
__global__ __launch_bounds__(256) void pack_t16_kernel(const void* __restrict__ in, int R, int Cn,
                                                       int64_t in_expert_stride, int half, bool gate_up,
                                                       uint16_t* __restrict__ out, int64_t out_rows, int out_ld) {
  __shared__ uint16_t tile[64][72];  // [input col][input row], rows padded to 144 B
  const int e = blockIdx.z;
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int tid = threadIdx.x;
  // load: thread -> (row r0 + tid/8 + 32 i, cols c0 + 8 (tid%8) .. +8), i = 0, 1
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int rr = tid / 8 + 32 * i, cc = 8 * (tid % 8);
    const int r = r0 + rr, c = c0 + cc;
    uint16_t v[8];
    const int64_t off = (int64_t)e * in_expert_stride + (int64_t)r * Cn + c;
    if (r < R && c + 8 <= Cn && off % (IN_F32 ? 4 : 8) == 0) {
      if (IN_F32) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(in) + off);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(in) + off + 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[q] = f32_to_bf16(a[q]);
          v[4 + q] = f32_to_bf16(b[q]);
        }
      } else {
        const i32x4_t a = *reinterpret_cast<const i32x4_t*>(static_cast<const uint16_t*>(in) + off);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[2 * q] = (uint16_t)((uint32_t)a[q] & 0xffffu);
          v[2 * q + 1] = (uint16_t)((uint32_t)a[q] >> 16);
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int cq = c + q;
        float f = 0.0f;
        if (r < R && cq < Cn) {
          const int64_t off = (int64_t)e * in_expert_stride + (int64_t)r * Cn + cq;
          f = IN_F32 ? static_cast<const float*>(in)[off] : bf16_to_f32(static_cast<const uint16_t*>(in)[off]);
        }
        v[q] = f32_to_bf16(f);
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) tile[cc + q][rr] = v[q];
  }
  __syncthreads();
  // store: thread -> (output row for input col c0 + tid/8 + 32 i, 8 elements r0 + 8 (tid%8))
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int cc = tid / 8 + 32 * i, rr = 8 * (tid % 8);
    const int c = c0 + cc, r = r0 + rr;
    if (c >= Cn || r >= R) continue;
    const int64_t orow = gate_up ? (int64_t)(c / 128) * 256 + half * 128 + (c % 128) : (int64_t)c;
    uint16_t* dst = out + ((int64_t)e * out_rows + orow) * out_ld + r;
    if (r + 8 <= R) {
      i32x4_t w;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        w[q] = (int)((uint32_t)tile[cc][rr + 2 * q] | ((uint32_t)tile[cc][rr + 2 * q + 1] << 16));
      *reinterpret_cast<i32x4_t*>(dst) = w;
    } else {
      for (int q = 0; r + q < R; ++q) dst[q] = tile[cc][rr + q];
    }
  }
}

// Zeroes what pack_t16_kernel leaves: in every packed row the elements [valid_cols,
// out_ld), and the whole rows that no input column maps to.  PAD_LANES neighbouring threads
// per row store 8 bytes each side by side (one thread per row stored a 128-byte pad as 16
// single stores, each instruction touching 64 rows); a pad that does not start at an 8-byte
// boundary (valid_cols % 4 != 0) is first finished element by element.  d 2048, F 2816, 16
// experts, w13 and w3 together: 16.9 -> 11.4 us.
constexpr int PAD_LANES = 16;
inline dim3 pad_grid(int64_t n_rows) { return dim3((unsigned)kmoe::ceil_div<int64_t>(n_rows * PAD_LANES, 256)); }
__global__ __launch_bounds__(256) void pack_pad_kernel(uint16_t* __restrict__ out, int64_t n_rows, int out_ld,
                                                       int valid_cols, int rows_per_expert, int valid_in_cols,
                                                       bool gate_up) {
  const int64_t row = (int64_t)blockIdx.x * (256 / PAD_LANES) + threadIdx.x / PAD_LANES;
  if (row >= n_rows) return;
  const int lane = threadIdx.x % PAD_LANES;
  const int pr = (int)(row % rows_per_expert);
  // the input column this packed row holds (gate_up: w1 / w2 column f of block f/128)
  const int c = gate_up ? (pr / 256) * 128 + (pr % 128) : pr;
  uint16_t* p = out + row * out_ld;
  const int from = c >= valid_in_cols ? 0 : valid_cols;
  const int whole = (from + 3) & ~3;
  if (from + lane < min(whole, out_ld)) p[from + lane] = 0;
  uint64_t* w = reinterpret_cast<uint64_t*>(p);
  for (int i = whole / 4 + lane; i < out_ld / 4; i += PAD_LANES) w[i] = 0ull;
}

// Backward packed layouts (rows K-contiguous, WPAD bytes after every row, zero padded):
//   mode ROWS_W3N : (E, round_up(F, 256), d)        row f = w3[e][f][:]      (dh = dY . w3^T, K = d)
//   mode ROWS_W13T: (E, round_up(d, 256), 2*F_pad)  row i = w1[e][i][:], w2[e][i][:] interleaved per 128
//                                                    columns like w13's rows  (dX = [dg|du] . w13, K = 2*F_pad)
//   mode ROWS_W1N : (E, round_up(d, 256), F_pad)    row i = w1[e][i][:]      (non-gated experts: dX = dp . w1^T)
// All are row copies with the columns rearranged (no transpose), 16 bytes per access;
// rows past F (w3n) or d (w13t, w1n) and the pads are written as zeros.
enum { ROWS_W3N = 0, ROWS_W13T = 1, ROWS_W1N = 2 };
template <bool IN_F32>
__global__ __launch_bounds__(256) void pack_rows16_kernel(const void* __restrict__ w1, const void* __restrict__ w2,
                                                          const void* __restrict__ w3, int d, int F, int mode,
                                                          uint16_t* __restrict__ out, int64_t out_rows, int out_ld,
                                                          int E) {
  const int nv = out_ld / 8;  // 16-byte vectors per packed row
  const int64_t n = (int64_t)E * out_rows * nv;
  const int Fp = round_up(F, 128);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t grow = i / nv;
    const int v = (int)(i - grow * nv);
    const int e = (int)(grow / out_rows);
    const int64_t row = grow - (int64_t)e * out_rows;
    const int c = 8 * v;  // first packed column of the vector
    const void* src = nullptr;
    int64_t off = 0;
    int n_ok = 0;  // source elements that exist (the rest are zero)
    if (mode == ROWS_W13T) {
      if (row < d && c < 2 * Fp) {
        const int half = (c >> 7) & 1, f = (c >> 8) * 128 + (c & 127);
        src = half ? w2 : w1;
        off = ((int64_t)e * d + row) * F + f;
        n_ok = F - f < 8 ? (F - f > 0 ? F - f : 0) : 8;
      }
    } else if (mode == ROWS_W1N) {
      if (row < d && c < Fp) {
        src = w1;
        off = ((int64_t)e * d + row) * F + c;
        n_ok = F - c < 8 ? (F - c > 0 ? F - c : 0) : 8;
      }
    } else if (row < F && c < d) {
      src = w3;
      off = ((int64_t)e * F + row) * d + c;
      n_ok = d - c < 8 ? d - c : 8;
    }
    i32x4_t wv = {0, 0, 0, 0};
    if (n_ok == 8 && (off % (IN_F32 ? 4 : 8)) == 0) {
      if (IN_F32) {
        const float* p = static_cast<const float*>(src) + off;
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          wv[q] = (int)((uint32_t)f32_to_bf16(a[2 * q]) | ((uint32_t)f32_to_bf16(a[2 * q + 1]) << 16));
          wv[2 + q] = (int)((uint32_t)f32_to_bf16(b[2 * q]) | ((uint32_t)f32_to_bf16(b[2 * q + 1]) << 16));
        }
      } else {
        wv = *reinterpret_cast<const i32x4_t*>(static_cast<const uint16_t*>(src) + off);
      }
    } else {
      uint16_t t[8];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        t[q] = q < n_ok ? (IN_F32 ? f32_to_bf16(static_cast<const float*>(src)[off + q])
                                  : static_cast<const uint16_t*>(src)[off + q])
                        : (uint16_t)0;
#pragma unroll
      for (int q = 0; q < 4; ++q) wv[q] = (int)((uint32_t)t[2 * q] | ((uint32_t)t[2 * q + 1] << 16));
    }
    *reinterpret_cast<i32x4_t*>(out + grow * out_ld + c) = wv;
  }
}

// Per-row fp8 quantisation of a bf16 matrix: each wave takes rows w, w + W, ... (W waves
// in the grid) and loads its next row into a second register set before it reduces and
// stores the current one, so a wave's reads and writes overlap (one row per wave, all
// resident at once, read every row first and wrote them all after).  NV: 16-byte vectors
// per lane of a row (the register sets are sized for the row, not for the largest one).
// PREFETCH = false (rows of more than 8 vectors per lane, where two register sets leave one
// wave per SIMD): one row per wave, no second set.
template <int NV, bool PREFETCH = true>
__global__ __launch_bounds__(256) void quant_rows_kernel(const uint16_t* __restrict__ in, int64_t rows,
                                                         const int32_t* __restrict__ n_rows_dev, int cols,
                                                         uint8_t* __restrict__ out, float* __restrict__ scale) {
  struct Regs {
    i32x4_t v[NV];
  };
  const int lane = threadIdx.x & 63;
  const int64_t nw = (int64_t)gridDim.x * 4;
  int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  int64_t nr = rows;
  if (n_rows_dev) nr = min<int64_t>(nr, (int64_t)*n_rows_dev);
  const int nvec = cols / 8;  // <= 64 * NV (chosen on the host)
  auto load = [&](int64_t row, Regs& rr) {
    const i32x4_t* src = reinterpret_cast<const i32x4_t*>(in + row * cols);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = lane + 64 * i;
      if (v < nvec) rr.v[i] = src[v];
    }
  };
  auto finish = [&](int64_t row, const Regs& rr) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (lane + 64 * i < nvec) {
#pragma unroll
        for (int q = 0; q < 4; ++q) amax = fmaxf(amax, bf16_pair_absmax((uint32_t)rr.v[i][q]));
      }
    amax = wave_max(amax);
    const float inv = amax > 0.0f ? 448.0f / amax : 0.0f;
    uint32_t* dst = reinterpret_cast<uint32_t*>(out + row * cols);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = lane + 64 * i;
      if (v < nvec) {
        uint32_t lo, hi;
        quant_vec_e4m3(rr.v[i], inv, lo, hi);
        *reinterpret_cast<uint2*>(dst + 2 * v) = make_uint2(lo, hi);
      }
    }
    if (lane == 0) scale[row] = amax / 448.0f;
  };
  Regs a;
  if constexpr (!PREFETCH) {
    if (r < nr) {
      load(r, a);
      finish(r, a);
    }
    return;
  }
  Regs b;
  if (r < nr) load(r, a);
  while (r < nr) {
    if (r + nw < nr) load(r + nw, b);
    finish(r, a);
    r += nw;
    if (r >= nr) break;
    if (r + nw < nr) load(r + nw, a);
    finish(r, b);
    r += nw;
  }
}

int elem_bytes(int dtype) { return dtype == KMOE_DTYPE_FP8_E4M3 ? 1 : 2; }

}  // namespace

extern "C" int kmoe_padded_ff(int F) { return round_up(F, 128); }

extern "C" size_t kmoe_packed_w13_bytes(int E, int d, int F, int dtype) {
  return (size_t)E * 2 * (size_t)round_up(F, 128) * ((size_t)d * (size_t)elem_bytes(dtype) + WPAD);
}

extern "C" size_t kmoe_packed_w3_bytes(int E, int d, int F, int dtype) {
  return (size_t)E * (size_t)round_up(d, 256) * ((size_t)round_up(F, 128) * (size_t)elem_bytes(dtype) + WPAD);
}

extern "C" int kmoe_pack_weights(const void* w1, const void* w2, const void* w3, int w_dtype, int E, int d, int F,
                                 int packed_dtype, void* w13_packed, float* w13_scale, void* w3_packed,
                                 float* w3_scale, void* stream) {
  KMOE_REQUIRE(w1 && w2 && w3 && w13_packed && w3_packed, KMOE_ERR_NULL, "kmoe_pack_weights: null buffer");
  KMOE_REQUIRE(E >= 1 && E <= KMOE_MAX_EXPERTS, KMOE_ERR_SHAPE, "kmoe_pack_weights: E=%d out of range", E);
  KMOE_REQUIRE(d > 0 && d % 64 == 0, KMOE_ERR_SHAPE, "kmoe_pack_weights: d=%d must be a positive multiple of 64", d);
  KMOE_REQUIRE(F > 0, KMOE_ERR_SHAPE, "kmoe_pack_weights: F=%d must be > 0", F);
  KMOE_REQUIRE(w_dtype == KMOE_DTYPE_BF16 || w_dtype == KMOE_DTYPE_F32, KMOE_ERR_DTYPE,
               "kmoe_pack_weights: weight dtype must be bf16 or f32");
  KMOE_REQUIRE(packed_dtype == KMOE_DTYPE_BF16 || packed_dtype == KMOE_DTYPE_FP8_E4M3, KMOE_ERR_DTYPE,
               "kmoe_pack_weights: packed dtype must be bf16 or fp8_e4m3");
  const bool fp8 = packed_dtype == KMOE_DTYPE_FP8_E4M3;
  KMOE_REQUIRE(!fp8 || (w13_scale && w3_scale), KMOE_ERR_NULL, "kmoe_pack_weights: fp8 needs scale buffers");
  hipStream_t s = kmoe::as_stream(stream);
  const int Fp = round_up(F, 128), dp = round_up(d, 256);
  const int64_t rows13 = 2 * (int64_t)Fp, rows3 = dp;
  const bool f32 = w_dtype == KMOE_DTYPE_F32;
  if (!fp8) {
    // bf16: vectorised transposes, then zeros in the pads and padding rows only
    const int ld13 = d + WPAD / 2, ld3 = Fp + WPAD / 2;
    uint16_t* o13 = static_cast<uint16_t*>(w13_packed);
    uint16_t* o3 = static_cast<uint16_t*>(w3_packed);
    const dim3 g13((unsigned)kmoe::ceil_div(F, 64), (unsigned)kmoe::ceil_div(d, 64), (unsigned)E);
    const dim3 g3((unsigned)kmoe::ceil_div(d, 64), (unsigned)kmoe::ceil_div(F, 64), (unsigned)E);
#define KMOE_PACK16(F32_)                                                                                         \
  do {                                                                                                            \
    hipLaunchKernelGGL(pack_t16_kernel<F32_>, g13, dim3(256), 0, s, w1, d, F, (int64_t)d * F, 0, true, o13, rows13, \
                       ld13);                                                                                     \
    hipLaunchKernelGGL(pack_t16_kernel<F32_>, g13, dim3(256), 0, s, w2, d, F, (int64_t)d * F, 1, true, o13, rows13, \
                       ld13);                                                                                     \
    hipLaunchKernelGGL(pack_t16_kernel<F32_>, g3, dim3(256), 0, s, w3, F, d, (int64_t)d * F, 0, false, o3, rows3,  \
                       ld3);                                                                                      \
  } while (0)
    if (f32)
      KMOE_PACK16(true);
    else
      KMOE_PACK16(false);
#undef KMOE_PACK16
    hipLaunchKernelGGL(pack_pad_kernel, pad_grid((int64_t)E * rows13), dim3(256), 0, s, o13,
                       (int64_t)E * rows13, ld13, d, (int)rows13, F, true);
    hipLaunchKernelGGL(pack_pad_kernel, pad_grid((int64_t)E * rows3), dim3(256), 0, s, o3,
                       (int64_t)E * rows3, ld3, F, (int)rows3, d, false);
    return kmoe::check_launch("kmoe_pack_weights");
  }
  // fp8: zero the padding (whole buffers: simple; the fp8 pack runs once per weight version)
  hipLaunchKernelGGL(zero_kernel, dim3(1024), dim3(256), 0, s, static_cast<uint8_t*>(w13_packed),
                     (int64_t)kmoe_packed_w13_bytes(E, d, F, packed_dtype));
  hipLaunchKernelGGL(zero_kernel, dim3(1024), dim3(256), 0, s, static_cast<uint8_t*>(w3_packed),
                     (int64_t)kmoe_packed_w3_bytes(E, d, F, packed_dtype));
  if (fp8) {
    hipLaunchKernelGGL(zero_f32_kernel, dim3(64), dim3(256), 0, s, w13_scale, (int64_t)E * rows13);
    hipLaunchKernelGGL(zero_f32_kernel, dim3(64), dim3(256), 0, s, w3_scale, (int64_t)E * rows3);
    const dim3 g13((unsigned)kmoe::ceil_div(F, 256), (unsigned)kmoe::ceil_div(d, COLS_ROWS), (unsigned)E);
    const dim3 g3((unsigned)kmoe::ceil_div(d, 256), (unsigned)kmoe::ceil_div(F, COLS_ROWS), (unsigned)E);
    if (f32) {
      hipLaunchKernelGGL(col_scale_kernel<true>, g13, dim3(256), 0, s, w1, d, F, (int64_t)d * F, 0, true, w13_scale, rows13);
      hipLaunchKernelGGL(col_scale_kernel<true>, g13, dim3(256), 0, s, w2, d, F, (int64_t)d * F, 1, true, w13_scale, rows13);
      hipLaunchKernelGGL(col_scale_kernel<true>, g3, dim3(256), 0, s, w3, F, d, (int64_t)d * F, 0, false, w3_scale, rows3);
    } else {
      hipLaunchKernelGGL(col_scale_kernel<false>, g13, dim3(256), 0, s, w1, d, F, (int64_t)d * F, 0, true, w13_scale, rows13);
      hipLaunchKernelGGL(col_scale_kernel<false>, g13, dim3(256), 0, s, w2, d, F, (int64_t)d * F, 1, true, w13_scale, rows13);
      hipLaunchKernelGGL(col_scale_kernel<false>, g3, dim3(256), 0, s, w3, F, d, (int64_t)d * F, 0, false, w3_scale, rows3);
    }
  }
  // w1/w2: (E, d, F) -> rows f, cols d.  w3: (E, F, d) -> rows n, cols f.
  const int eb = elem_bytes(packed_dtype);
  const int ld13 = d + WPAD / eb, ld3 = Fp + WPAD / eb;  // packed row strides in elements
  const dim3 gt13((unsigned)kmoe::ceil_div(F, 64), (unsigned)kmoe::ceil_div(d, 64), (unsigned)E);
  const dim3 gt3((unsigned)kmoe::ceil_div(d, 64), (unsigned)kmoe::ceil_div(F, 64), (unsigned)E);
  uint8_t* o13 = static_cast<uint8_t*>(w13_packed);
  uint8_t* o3 = static_cast<uint8_t*>(w3_packed);
#define KMOE_PACK(F32_, FP8_)                                                                                        \
  do {                                                                                                               \
    hipLaunchKernelGGL((pack_transpose_kernel<F32_, FP8_>), gt13, dim3(256), 0, s, w1, d, F, (int64_t)d * F, 0, true, \
                       o13, rows13, ld13, w13_scale);                                                                   \
    hipLaunchKernelGGL((pack_transpose_kernel<F32_, FP8_>), gt13, dim3(256), 0, s, w2, d, F, (int64_t)d * F, 1, true, \
                       o13, rows13, ld13, w13_scale);                                                                   \
    hipLaunchKernelGGL((pack_transpose_kernel<F32_, FP8_>), gt3, dim3(256), 0, s, w3, F, d, (int64_t)d * F, 0, false, \
                       o3, rows3, ld3, w3_scale);                                                                     \
  } while (0)
  if (f32 && fp8)
    KMOE_PACK(true, true);
  else if (f32)
    KMOE_PACK(true, false);
  else if (fp8)
    KMOE_PACK(false, true);
  else
    KMOE_PACK(false, false);
#undef KMOE_PACK
  if (fp8) {
    hipLaunchKernelGGL(finalize_scale_kernel, dim3(64), dim3(256), 0, s, w13_scale, (int64_t)E * rows13);
    hipLaunchKernelGGL(finalize_scale_kernel, dim3(64), dim3(256), 0, s, w3_scale, (int64_t)E * rows3);
  }
  return kmoe::check_launch("kmoe_pack_weights");
}

extern "C" int kmoe_quant_rows_fp8(const void* in, int64_t rows, const int32_t* n_rows_dev, int cols, uint8_t* out,
                                   float* scale, void* stream) {
  KMOE_REQUIRE(in && out && scale, KMOE_ERR_NULL, "kmoe_quant_rows_fp8: null buffer");
  KMOE_REQUIRE(rows >= 0 && cols > 0 && cols % 8 == 0, KMOE_ERR_SHAPE, "kmoe_quant_rows_fp8: bad shape");
  KMOE_REQUIRE(cols <= 64 * 8 * ROW_REGS, KMOE_ERR_UNSUPPORTED, "kmoe_quant_rows_fp8: cols=%d > %d", cols,
               64 * 8 * ROW_REGS);
  if (rows == 0) return KMOE_OK;
  // up to 8 vectors per lane: as many workgroups per CU as are resident at once (the
  // kernel's register use for NV = 2, 4, 8: 7, 4, 3 waves per SIMD), each wave looping
  // over its rows; wider rows: one row per wave
  const int nv = kmoe::ceil_div(cols / 8, 64);
  const int per_cu = nv <= 2 ? 6 : nv <= 4 ? 4 : 3;
  const int64_t all_rows = kmoe::ceil_div<int64_t>(rows, 4);  // one row per wave
  const int64_t blocks = nv <= 8 ? std::min<int64_t>(all_rows, (int64_t)kmoe::cu_count() * per_cu) : all_rows;
  hipStream_t s = kmoe::as_stream(stream);
  const uint16_t* ip = static_cast<const uint16_t*>(in);
  if (nv <= 2)
    hipLaunchKernelGGL(quant_rows_kernel<2>, dim3((unsigned)blocks), dim3(256), 0, s, ip, rows, n_rows_dev, cols, out, scale);
  else if (nv <= 4)
    hipLaunchKernelGGL(quant_rows_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, s, ip, rows, n_rows_dev, cols, out, scale);
  else if (nv <= 8)
    hipLaunchKernelGGL(quant_rows_kernel<8>, dim3((unsigned)blocks), dim3(256), 0, s, ip, rows, n_rows_dev, cols, out, scale);
  else
    hipLaunchKernelGGL((quant_rows_kernel<ROW_REGS, false>), dim3((unsigned)blocks), dim3(256), 0, s, ip, rows,
                       n_rows_dev, cols, out, scale);
  return kmoe::check_launch("kmoe_quant_rows_fp8");
}

extern "C" size_t kmoe_packed_w3n_bytes(int E, int d, int F) {
  return (size_t)E * (size_t)round_up(F, 256) * ((size_t)d * 2 + WPAD);
}

extern "C" size_t kmoe_packed_w13t_bytes(int E, int d, int F) {
  return (size_t)E * (size_t)round_up(d, 256) * ((size_t)2 * round_up(F, 128) * 2 + WPAD);
}

extern "C" int kmoe_pack_weights_bwd(const void* w1, const void* w2, const void* w3, int w_dtype, int E, int d, int F,
                                     void* w3n_packed, void* w13t_packed, void* stream) {
  KMOE_REQUIRE(w1 && w2 && w3 && w3n_packed && w13t_packed, KMOE_ERR_NULL, "kmoe_pack_weights_bwd: null buffer");
  KMOE_REQUIRE(E >= 1 && E <= KMOE_MAX_EXPERTS, KMOE_ERR_SHAPE, "kmoe_pack_weights_bwd: E=%d out of range", E);
  KMOE_REQUIRE(d > 0 && d % 64 == 0, KMOE_ERR_SHAPE, "kmoe_pack_weights_bwd: d=%d must be a positive multiple of 64", d);
  KMOE_REQUIRE(F > 0, KMOE_ERR_SHAPE, "kmoe_pack_weights_bwd: F=%d must be > 0", F);
  KMOE_REQUIRE(w_dtype == KMOE_DTYPE_BF16 || w_dtype == KMOE_DTYPE_F32, KMOE_ERR_DTYPE,
               "kmoe_pack_weights_bwd: weight dtype must be bf16 or f32");
  hipStream_t s = kmoe::as_stream(stream);
  const bool f32 = w_dtype == KMOE_DTYPE_F32;
  const int Fp = round_up(F, 128);
  const int64_t r3 = round_up(F, 256), r13 = round_up(d, 256);
  const int ld3 = d + WPAD / 2, ld13 = 2 * Fp + WPAD / 2;
  if (f32) {
    hipLaunchKernelGGL(pack_rows16_kernel<true>, dim3(4096), dim3(256), 0, s, w1, w2, w3, d, F, (int)ROWS_W3N,
                       static_cast<uint16_t*>(w3n_packed), r3, ld3, E);
    hipLaunchKernelGGL(pack_rows16_kernel<true>, dim3(4096), dim3(256), 0, s, w1, w2, w3, d, F, (int)ROWS_W13T,
                       static_cast<uint16_t*>(w13t_packed), r13, ld13, E);
  } else {
    hipLaunchKernelGGL(pack_rows16_kernel<false>, dim3(4096), dim3(256), 0, s, w1, w2, w3, d, F, (int)ROWS_W3N,
                       static_cast<uint16_t*>(w3n_packed), r3, ld3, E);
    hipLaunchKernelGGL(pack_rows16_kernel<false>, dim3(4096), dim3(256), 0, s, w1, w2, w3, d, F, (int)ROWS_W13T,
                       static_cast<uint16_t*>(w13t_packed), r13, ld13, E);
  }
  return kmoe::check_launch("kmoe_pack_weights_bwd");
}

// ---- non-gated experts (silu(x . w1) . w2, moe.py:187-191,281-283): w1 (E, d, F), w2 (E, F, d)
extern "C" size_t kmoe_packed_w1t_bytes(int E, int d, int F) {
  return (size_t)E * (size_t)round_up(F, 256) * ((size_t)d * 2 + WPAD);
}

extern "C" size_t kmoe_packed_w1n_bytes(int E, int d, int F) {
  return (size_t)E * (size_t)round_up(d, 256) * ((size_t)round_up(F, 128) * 2 + WPAD);
}

static int check_plain_pack(const char* who, const void* w1, const void* w2, const void* o1, const void* o2,
                            int w_dtype, int E, int d, int F) {
  KMOE_REQUIRE(w1 && w2 && o1 && o2, KMOE_ERR_NULL, "%s: null buffer", who);
  KMOE_REQUIRE(E >= 1 && E <= KMOE_MAX_EXPERTS, KMOE_ERR_SHAPE, "%s: E=%d out of range", who, E);
  KMOE_REQUIRE(d > 0 && d % 64 == 0, KMOE_ERR_SHAPE, "%s: d=%d must be a positive multiple of 64", who, d);
  KMOE_REQUIRE(F > 0, KMOE_ERR_SHAPE, "%s: F=%d must be > 0", who, F);
  KMOE_REQUIRE(w_dtype == KMOE_DTYPE_BF16 || w_dtype == KMOE_DTYPE_F32, KMOE_ERR_DTYPE,
               "%s: weight dtype must be bf16 or f32", who);
  return KMOE_OK;
}

extern "C" int kmoe_pack_weights_plain(const void* w1, const void* w2, int w_dtype, int E, int d, int F,
                                       void* w1t_packed, void* w2t_packed, void* stream) {
  const int rc = check_plain_pack("kmoe_pack_weights_plain", w1, w2, w1t_packed, w2t_packed, w_dtype, E, d, F);
  if (rc) return rc;
  hipStream_t s = kmoe::as_stream(stream);
  const int Fp = round_up(F, 128);
  const int64_t r1 = round_up(F, 256), r2 = round_up(d, 256);
  const int ld1 = d + WPAD / 2, ld2 = Fp + WPAD / 2;
  uint16_t* o1 = static_cast<uint16_t*>(w1t_packed);
  uint16_t* o2 = static_cast<uint16_t*>(w2t_packed);
  // w1t: row f = w1[e][:, f] (K = d); w2t: row n = w2[e][:, n] (K = F_pad), the down pack's layout
  const dim3 g1((unsigned)kmoe::ceil_div(F, 64), (unsigned)kmoe::ceil_div(d, 64), (unsigned)E);
  const dim3 g2((unsigned)kmoe::ceil_div(d, 64), (unsigned)kmoe::ceil_div(F, 64), (unsigned)E);
  if (w_dtype == KMOE_DTYPE_F32) {
    hipLaunchKernelGGL(pack_t16_kernel<true>, g1, dim3(256), 0, s, w1, d, F, (int64_t)d * F, 0, false, o1, r1, ld1);
    hipLaunchKernelGGL(pack_t16_kernel<true>, g2, dim3(256), 0, s, w2, F, d, (int64_t)d * F, 0, false, o2, r2, ld2);
  } else {
    hipLaunchKernelGGL(pack_t16_kernel<false>, g1, dim3(256), 0, s, w1, d, F, (int64_t)d * F, 0, false, o1, r1, ld1);
    hipLaunchKernelGGL(pack_t16_kernel<false>, g2, dim3(256), 0, s, w2, F, d, (int64_t)d * F, 0, false, o2, r2, ld2);
  }
  hipLaunchKernelGGL(pack_pad_kernel, pad_grid((int64_t)E * r1), dim3(256), 0, s, o1,
                     (int64_t)E * r1, ld1, d, (int)r1, F, false);
  hipLaunchKernelGGL(pack_pad_kernel, pad_grid((int64_t)E * r2), dim3(256), 0, s, o2,
                     (int64_t)E * r2, ld2, F, (int)r2, d, false);
  return kmoe::check_launch("kmoe_pack_weights_plain");
}

extern "C" int kmoe_pack_weights_plain_bwd(const void* w1, const void* w2, int w_dtype, int E, int d, int F,
                                           void* w2n_packed, void* w1n_packed, void* stream) {
  const int rc = check_plain_pack("kmoe_pack_weights_plain_bwd", w1, w2, w2n_packed, w1n_packed, w_dtype, E, d, F);
  if (rc) return rc;
  hipStream_t s = kmoe::as_stream(stream);
  const int Fp = round_up(F, 128);
  const int64_t r2 = round_up(F, 256), r1 = round_up(d, 256);
  const int ld2 = d + WPAD / 2, ld1 = Fp + WPAD / 2;
  // w2n: row f = w2[e][f][:] (dh = dY . w2^T, K = d), the w3n layout of w2; w1n: row i = w1[e][i][:] (K = F_pad)
  if (w_dtype == KMOE_DTYPE_F32) {
    hipLaunchKernelGGL(pack_rows16_kernel<true>, dim3(4096), dim3(256), 0, s, w1, nullptr, w2, d, F, (int)ROWS_W3N,
                       static_cast<uint16_t*>(w2n_packed), r2, ld2, E);
    hipLaunchKernelGGL(pack_rows16_kernel<true>, dim3(4096), dim3(256), 0, s, w1, nullptr, w2, d, F, (int)ROWS_W1N,
                       static_cast<uint16_t*>(w1n_packed), r1, ld1, E);
  } else {
    hipLaunchKernelGGL(pack_rows16_kernel<false>, dim3(4096), dim3(256), 0, s, w1, nullptr, w2, d, F, (int)ROWS_W3N,
                       static_cast<uint16_t*>(w2n_packed), r2, ld2, E);
    hipLaunchKernelGGL(pack_rows16_kernel<false>, dim3(4096), dim3(256), 0, s, w1, nullptr, w2, d, F, (int)ROWS_W1N,
                       static_cast<uint16_t*>(w1n_packed), r1, ld1, E);
  }
  return kmoe::check_launch("kmoe_pack_weights_plain_bwd");
}
