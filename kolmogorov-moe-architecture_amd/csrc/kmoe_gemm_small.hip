// Grouped products with few rows per expert (decode steps, short prompts), bf16.
//
// There every expert's weights are read once for a handful of rows, so the product is bound
// by streaming the packed weights (a plain read of this size reaches 6.1 TB/s).  The
// 256-row tiles of kmoe_gemm_tile.h stream them through LDS, one workgroup per CU; here
// each wave loads its weight rows straight into MFMA operand registers, at four
// workgroups per CU (104 to 122 registers a lane).  d 2048, F 2816, 16 experts, top-2, weights
// not in a cache, 256-row tiles -> here: 96 rows, 6 an expert, gate/up 77.0 -> 66.1 us (5.6
// TB/s), down 39.7 -> 35.6 (5.2); one token, two experts, 21.5 -> 12.2 (3.8) and 25.9 -> 8.8
// (2.6), bound by latency.
//
// Operand fragments (v_mfma_f32_16x16x32_bf16, weights first): lane l holds row l % 16 of a
// 16-row block at the 8 K values of chunk l / 16, so one load instruction takes 64
// contiguous bytes of 16 rows and the two substeps of a 64-wide K-step a whole 128-byte
// line of each.  The result lane holds four consecutive output columns of one row.
#include "kmoe_gemm_tile.h"

using namespace kmoe_tiles;

namespace {

// (expert, first row, row end) of slot `slot` (SMALL_ROWS rows each, numbered expert by
// expert); false if there are fewer slots.
__device__ __forceinline__ bool small_slot(const int32_t* __restrict__ offsets, int E, int slot, int& e, int& m0,
                                           int& m_end) {
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = 0;
  if (lane < E) {
    lo = offsets[lane];
    hi = offsets[lane + 1];
  }
  int incl = (hi - lo + SMALL_ROWS - 1) / SMALL_ROWS;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  const uint64_t m = __ballot(slot < incl);
  if (!m) return false;
  e = __builtin_ctzll(m);
  const int before = e > 0 ? __builtin_amdgcn_readlane(incl, e - 1) : 0;
  m0 = __builtin_amdgcn_readlane(lo, e) + (slot - before) * SMALL_ROWS;
  m_end = __builtin_amdgcn_readlane(hi, e);
  return true;
}

// Activation row of permuted row r (GATHER: row_index[row_token[r]] or row_token[r]).
template <bool GATHER>
__device__ __forceinline__ int act_row(const GemmArgs& g, int r, int m0) {
  if constexpr (!GATHER) return r - m0;
  const int t = g.row_token[r];
  return g.row_index ? g.row_index[t] : t;
}

__device__ __forceinline__ bf16x8_t load_frag(__amdgpu_buffer_rsrc_t rs, uint32_t off, int soff) {
  return __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rs, off, soff, 0));
}

// Four output columns of one row from the gate and up sums of that row (gate/up), stored
// as 8 bytes; SAVE_GU also stores the pre-activation values in the packed column order.
// f: first of the four columns.
template <bool SAVE_GU, bool RSCALE>
__device__ __forceinline__ void put_gate_up(const GemmArgs& g, int row, int f, f32x4_t gate, f32x4_t up) {
  if constexpr (RSCALE) {
    const float s = g.a_scale[g.row_token[row]];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      gate[c] *= s;
      up[c] *= s;
    }
  }
  float v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = silu_fast_f32(gate[c]) * up[c];
  *reinterpret_cast<i32x2_t*>(g.C + (int64_t)row * g.ldc + f) = pack4_bf16(v[0], v[1], v[2], v[3]);
  if constexpr (SAVE_GU) {
    uint16_t* p = g.gu_out + (int64_t)row * 2 * g.ldc + (f >> 7) * 256 + (f & 127);
    *reinterpret_cast<i32x2_t*>(p) = pack4_bf16(gate[0], gate[1], gate[2], gate[3]);
    *reinterpret_cast<i32x2_t*>(p + 128) = pack4_bf16(up[0], up[1], up[2], up[3]);
  }
}

// A workgroup owns one slot and 32 weight rows (gate/up: 16 gate and the
// 16 up rows of the same columns).  Its four waves split K, each with its rows' and its
// weights' K range to itself, so nothing is shared until the four partial sums are added
// in wave order through LDS.
// Two K-steps in flight per wave: more, at fewer waves per CU, stream slower (gate/up of 96
// rows over 16 experts, d 2048, F 2816, in one run: 1 step 67.1 us, 2 67.6, 3 73.2, 4 75.7, 8
// 97.0).  Interleaving the waves' steps, eight waves per workgroup and
// non-temporal weight loads were slower too.
constexpr int DEPTH = 2;
template <bool GATE_UP, bool GATHER, bool SAVE_GU, bool RSCALE, bool DUAL>
__global__ __launch_bounds__(256) void small_rows_kernel(GemmArgs g, const int32_t* __restrict__ offsets, int E, int n_ct) {
  __shared__ f32x4_t red[4][4][64];
  const int slot = blockIdx.x / n_ct, ct = blockIdx.x - slot * n_ct;
  int e, m0, m_end;
  if (!small_slot(offsets, E, slot, e, m0, m_end)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, lq = lane >> 4;
  const int rows = min(m_end - m0, SMALL_ROWS);
  const int nk = g.k_bytes / KB;
  const int s0 = wave * nk / 4, s1 = (wave + 1) * nk / 4;

  const uint8_t* const bbase = g.B + (int64_t)e * g.b_expert_rows * g.ldb_bytes;
  const uint8_t* const b2base = DUAL ? g.B2 + (int64_t)e * g.b_expert_rows * g.ldb_bytes : nullptr;
  const uint8_t* const abase = GATHER ? g.A : g.A + (int64_t)m0 * g.lda_bytes;
  uint32_t boff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = GATE_UP ? (ct >> 3) * 256 + j * 128 + (ct & 7) * 16 + r16 : ct * 32 + j * 16 + r16;
    boff[j] = (uint32_t)row * (uint32_t)g.ldb_bytes + lq * 16u;
  }
  f32x4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  auto run = [&](auto mb_tag) {
    constexpr int MB = decltype(mb_tag)::value;
    bf16x8_t b[DEPTH][2][2], a[DEPTH][2][MB];
    // step s into ring entry u; steps past the wave's range read nothing (empty window)
    auto load_b = [&](int u, int s) {
      const uint8_t* const base = DUAL && dual_step_second(s) ? b2base : bbase;
      const __amdgpu_buffer_rsrc_t rs = make_rsrc_window(base, s < s1 ? 0x7fffffff : 0);
      const int soff = DUAL ? dual_step_offset(s) : s * KB;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) b[u][i][j] = load_frag(rs, boff[j] + 64u * i, soff);
    };
    uint32_t aoff[MB];
    auto load_a = [&](int u, int s) {
      const __amdgpu_buffer_rsrc_t rs = make_rsrc_window(abase, s < s1 ? 0x7fffffff : 0);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 2; ++i) a[u][i][mb] = load_frag(rs, aoff[mb] + 64u * i, s * KB);
    };
    // the weights first: their addresses do not wait for the row lookup
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) load_b(u, s0 + u);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int r = mb * 16 + r16;
      aoff[mb] = r < rows ? (uint32_t)act_row<GATHER>(g, m0 + r, m0) * (uint32_t)g.lda_bytes + lq * 16u : 0x80000000u;
    }
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) load_a(u, s0 + u);
    for (int s = s0; s < s1; s += DEPTH) {
#pragma unroll
      for (int u = 0; u < DEPTH; ++u) {
        // entries past the range hold zeros
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[mb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[u][i][j], a[u][i][mb], acc[mb][j], 0, 0, 0);
        load_b(u, s + u + DEPTH);
        load_a(u, s + u + DEPTH);
      }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < 2; ++j) red[wave][mb * 2 + j][lane] = acc[mb][j];
  };
  const int nb = rows > 16 ? 2 : 1;
  if (nb == 2)
    run(std::integral_constant<int, 2>{});
  else
    run(std::integral_constant<int, 1>{});
  __syncthreads();
  auto total = [&](int blk) {
    f32x4_t t = red[0][blk][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) t += red[w][blk][lane];
    return t;
  };
  if constexpr (GATE_UP) {
    const int row = wave * 16 + r16, f = ct * 16 + 4 * lq;
    if (wave < nb && row < rows) put_gate_up<SAVE_GU, RSCALE>(g, m0 + row, f, total(2 * wave), total(2 * wave + 1));
  } else {
    const int row = (wave >> 1) * 16 + r16, col = ct * 32 + (wave & 1) * 16 + 4 * lq;
    if (wave < 2 * nb && row < rows && col < g.n_valid) {
      const f32x4_t t = total(wave);
      *reinterpret_cast<i32x2_t*>(g.C + (int64_t)(m0 + row) * g.ldc + col) = pack4_bf16(t[0], t[1], t[2], t[3]);
    }
  }
}

template <bool GATE_UP, bool GATHER, bool SAVE_GU, bool RSCALE, bool DUAL = false>
void launch_small(const GemmLaunch& l) {
  hipLaunchKernelGGL((small_rows_kernel<GATE_UP, GATHER, SAVE_GU, RSCALE, DUAL>), dim3(l.blocks), dim3(256), 0, l.s, l.g,
                     l.offsets, l.E, l.n_tiles);
}

}  // namespace

namespace kmoe_tiles {

void launch_small_rows(const GemmLaunch& l, bool gate_up) {
  if (l.g.B2)
    launch_small<false, false, false, false, true>(l);
  else if (!gate_up)
    launch_small<false, false, false, false>(l);
  else if (!l.g.row_token)
    launch_small<true, false, false, false>(l);
  else if (l.g.gu_out)
    launch_small<true, true, true, false>(l);
  else if (l.g.a_scale)
    launch_small<true, true, false, true>(l);
  else
    launch_small<true, true, false, false>(l);
}

}  // namespace kmoe_tiles
