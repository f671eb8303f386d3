// Grouped SwiGLU expert GEMMs on CDNA4 MFMA: the tile kernels.
// Replaces moe_kernels.grouped_swiglu_forward (moe_arch/kernels/grouped_gemm.cu:186-257)
// and the padded bmm block of GroupedExperts.forward (moe_arch/model/moe.py:275-279):
//   gate_up:  h[r, f] = silu(x[r] . w1[e][:, f]) * (x[r] . w2[e][:, f])     (ffn.py:17-64)
//   down:     y[r, n] = h[r] . w3[e][:, n]
// for the rows r of expert e, [offsets[e], offsets[e+1]).
//
// Tiling: a workgroup of 4 waves (one per SIMD) owns a 256-row x 256-B-row tile;
// waves form 2 (rows) x 2 (B rows) and each computes 128 x 128, 256 fp32 accumulators
// per lane: bf16 as 8x8 blocks of v_mfma_f32_16x16x32_bf16, fp8 as 4x4 blocks of
// v_mfma_scale_f32_32x32x64_f8f6f4.  (The expert GEMMs run at the chip's power limit,
// and on random data the 16x16x32 bf16 form sustains a higher clock than 32x32x16:
// 0.81 against 0.70 of the bf16 peak in an MFMA-only loop; the fp8 16x16x128 form runs
// at half rate, so fp8 keeps 32x32x64.)  A 128x128 wave tile reads 0.5 KiB of LDS per
// 32 K-MACs of output, the least a 4-wave workgroup of this tile allows.  K advances 64
// bf16 (128 fp8 bytes) per pipeline step through 2 LDS stages of 2 x 32 KiB.  Tile
// data is loaded into registers with buffer loads (the K offset is a scalar operand)
// one step ahead and written to the stage not being read, 16-byte chunks XOR-swizzled
// so that both the 1 KiB block writes and every 16-lane fragment read pass are
// bank-conflict free.  bf16: the K loop is emitted in program order (each MFMA with
// the LDS or memory instruction assigned to it); fp8: interleaved by scheduling
// groups, fragments double buffered.  One barrier per step.
// The MFMAs take the B fragment as their first operand, so each lane accumulates
// runs of four consecutive output columns of one row; the epilogue packs them to
// 8-byte bf16 runs in registers, stages the tile through LDS and writes it with
// 16-byte row stores (full e4m3 tiles: merged across lanes and stored from registers).
//
// Ragged groups: every row tile ("slot") of every expert is enumerated from the
// device-resident offsets; the grid is sized for the worst case
// (ceil(max_rows/256) + E slots) and workgroups without a tile exit (full e4m3 tiles: one
// workgroup per CU loops over its tiles).  No host sync.
// Tile order is XCD-aware: workgroups are dispatched round-robin over the 8 XCDs,
// so consecutive ids of one XCD are given 32-tile super-blocks of 4 slots x 8
// column tiles, which then share their A and B K-slices in that XCD's L2.
//
// Weights are consumed in a packed, derived layout (kmoe_pack_weights):
//   w13: (E, 2*F_pad, d)   per 128-wide f block: 128 gate rows then 128 up rows,
//                          each row K(=d)-contiguous (w1/w2 transposed)
//   w3 : (E, d_pad, F_pad) row n K(=f)-contiguous (w3 transposed), d_pad = round_up(d, 256)
// Every packed row is followed by WPAD bytes of padding: with power-of-two row
// strides the 256 rows of a tile K-slice would all map to the same memory
// channels; the pad spreads them (measured: +20% on the gate/up GEMM).
#pragma once

#include <type_traits>

#include "kmoe_common.h"

namespace kmoe_tiles {

constexpr int BM = 256;
constexpr int BN = 256;       // B rows per tile (gate_up: 128 gate + 128 up)
constexpr int GEMM_THREADS = 256;
constexpr int WPAD = 128;     // bytes of padding after every packed weight row
constexpr int NXCD = 8;
constexpr int SB_TILES = 32;  // tiles per XCD super-block (4 slots x 8 column tiles)
constexpr int KB = 128;       // K bytes per row per pipeline step (64 bf16 / 128 fp8)
constexpr int TB = BM * KB;   // bytes of one A or B stage tile (32 KiB)
constexpr int NST = 2;        // LDS stages: one read while the next is written
constexpr int CPR = KB / 16;  // 16-byte chunks per tile row
constexpr int RPB = 1024 / KB;                        // tile rows per 1 KiB load block
constexpr int BLK_PER_WAVE = (BM * KB / 1024) / 4;    // load blocks per wave per operand per step
// output staging: 256 rows x up to 256 bf16 columns, rows padded by 16 bytes
constexpr int OUT_STRIDE_MAX = 256 * 2 + 16;
constexpr int SCALE_LDS = (NST * 2 * TB > BM * OUT_STRIDE_MAX) ? NST * 2 * TB : BM * OUT_STRIDE_MAX;
// fp8: the tile's A-row and B-row scales (256 floats each) after the stages / output staging
constexpr int GEMM_LDS = SCALE_LDS + 8 * 1024;
static_assert(GEMM_LDS <= 160 * 1024, "LDS budget");

// Byte offset of 16-byte chunk `chunk` of tile row `row`.  A 128-byte row puts rows
// r and r+2 on the same banks; XOR-ing the chunk by (row/2)%8 gives the 16 lanes of
// an LDS read pass (16 consecutive rows, one chunk) 16 distinct 16-byte bank groups.
__device__ __forceinline__ int swz(int row, int chunk) { return row * KB + ((chunk ^ ((row >> 1) & (CPR - 1))) << 4); }

__host__ __device__ inline int round_up(int a, int b) { return (a + b - 1) / b * b; }

// Row slots.  Lane e of a wave holds the row range [lo, hi) of expert e (E <= 64)
// and its number of 256-row slots; slots are numbered expert by expert.
struct SlotTable {
  int lo, hi, ns;  // this lane's expert
  int n_slots;     // all experts (wave-uniform)
};
__device__ __forceinline__ SlotTable load_slots(const int32_t* __restrict__ offsets, int E) {
  const int lane = threadIdx.x & 63;
  SlotTable t;
  t.lo = 0;
  t.hi = 0;
  if (lane < E) {
    t.lo = offsets[lane];
    t.hi = offsets[lane + 1];
  }
  t.ns = (t.hi - t.lo + BM - 1) / BM;
  int n = t.ns;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  t.n_slots = __builtin_amdgcn_readfirstlane(n);
  return t;
}
// (expert, first row, row end) of slot `slot` < n_slots: a readlane walk over the
// experts' slot counts.
__device__ __forceinline__ void find_slot(const SlotTable& t, int E, int slot, int& e_out, int& m0, int& m_end) {
  int base = 0;
  e_out = 0;
  m0 = 0;
  m_end = 0;
  for (int e = 0; e < E; ++e) {
    const int n = __builtin_amdgcn_readlane(t.ns, e);
    if (slot < base + n) {
      e_out = e;
      m0 = __builtin_amdgcn_readlane(t.lo, e) + (slot - base) * BM;
      m_end = __builtin_amdgcn_readlane(t.hi, e);
      return;
    }
    base += n;
  }
}

// Dense tile order: slots in groups of 4, each group enumerated column tile by
// column tile (4 consecutive tiles share a column tile, so 32 consecutive tiles are
// 8 column tiles x 4 slots); the last, partial group likewise with its slots.
__device__ __forceinline__ void dense_tile(int t, int n_slots, int n_tiles, int& slot, int& nt) {
  const int full = (n_slots >> 2) * 4 * n_tiles;
  if (t < full) {
    const int g = t / (4 * n_tiles), r = t - g * 4 * n_tiles;
    nt = r >> 2;
    slot = g * 4 + (r & 3);
  } else {
    const int rem = n_slots & 3, u = t - full;
    nt = u / rem;
    slot = (n_slots & ~3) + (u - nt * rem);
  }
}

// Workgroup id L < n (n a multiple of 256) -> dense tile, XCD-aware: workgroups are
// dispatched round-robin over the 8 XCDs, so the consecutive ids one XCD receives
// are given 32-tile super-blocks, which share A and B K-slices in that XCD's L2.
__device__ __forceinline__ int xcd_tile(int L) {
  const int xcd = L % NXCD, i = L / NXCD;
  return ((i / SB_TILES) * NXCD + xcd) * SB_TILES + (i % SB_TILES);
}

template <bool FP8>
struct Frag;
template <>
struct Frag<false> {
  bf16x8_t v;
};
template <>
struct Frag<true> {
  i32x8_t v;
};

// One e4m3 MFMA operand fragment of K-substep `i` (64 of K, chunks 4i+2lh and 4i+2lh+1) for
// LDS tile row `r`.
__device__ __forceinline__ void read_frag(const uint8_t* l, int r, int i, int lh, Frag<true>& f) {
  const int ch = 4 * i + 2 * lh;
  const i32x4_t lo = *reinterpret_cast<const i32x4_t*>(l + swz(r, ch));
  const i32x4_t hi = *reinterpret_cast<const i32x4_t*>(l + swz(r, ch + 1));
  f.v = i32x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

__device__ __forceinline__ void mfma(f32x16_t& acc, const Frag<true>& a, const Frag<true>& b) {
  acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a.v, b.v, acc, 0, 0, 0, 127, 0, 127);
}

// bf16 tiles run on v_mfma_f32_16x16x32_bf16: on random data the 32x32x16 form holds the
// chip at 0.70 of the bf16 peak under its power limit (an MFMA-only loop, all CUs), the
// 16x16x32 form at 0.81 (it moves half the accumulator bytes per FLOP).  Fragment of
// K-substep `i` (32 of K: chunks 4i .. 4i+3) for LDS tile rows r0 .. r0+15: lane l reads
// row r0 + l%16 (`r`), chunk 4i + l/16 (`lq`); a 16-lane pass is 16 consecutive rows of
// one logical chunk, which the swizzle spreads over all banks.
__device__ __forceinline__ void read_frag16(const uint8_t* l, int r, int i, int lq, Frag<false>& f) {
  f.v = *reinterpret_cast<const bf16x8_t*>(l + swz(r, 4 * i + lq));
}
__device__ __forceinline__ void mfma16(f32x4_t& acc, const Frag<false>& a, const Frag<false>& b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc, 0, 0, 0);
}

// B-tile geometry of a tile whose waves hold WNB 32-row B blocks each (WNB = 4: the
// full 256 B rows; 2 and 1: the narrow tiles of the split tail, a half or a
// quarter `q` of a full tile's output columns).  LDS B row of block j of wave
// column wn:  down: 32 WNB wn + 32 j + lr;  gate_up (WNB >= 2): the first WNB/2
// blocks are gate rows and the rest the up rows of the same f columns;  gate_up
// WNB = 1: the wave's one block is 16 gate rows then the 16 up rows of the same f
// columns (LDS rows 32 wn + lr).
template <bool GATE_UP, int WNB>
__device__ __forceinline__ int b_lds_row(int wn, int j, int lr) {
  if constexpr (GATE_UP && WNB == 1) {
    return wn * 32 + lr;
  } else if constexpr (GATE_UP) {
    constexpr int H = WNB / 2;
    return (j / H) * (32 * WNB) + wn * (16 * WNB) + (j % H) * 32 + lr;
  } else {
    return wn * (32 * WNB) + j * 32 + lr;
  }
}
// Row of the 256-row packed B tile that LDS B row `lrow` holds (identity for WNB = 4).
// gate_up packs 128 gate rows then 128 up rows per full tile.
template <bool GATE_UP, int WNB>
__device__ __forceinline__ int b_packed_row(int lrow, int q) {
  if constexpr (GATE_UP && WNB == 1) {
    const int i = lrow & 31;  // f column 32 q + 16 (lrow / 32) + i % 16; up rows from i = 16
    return (i >> 4) * 128 + q * 32 + (lrow >> 5) * 16 + (i & 15);
  } else if constexpr (GATE_UP) {
    constexpr int HR = 32 * WNB;  // gate (or up) rows of the tile
    return (lrow / HR) * 128 + q * HR + lrow % HR;
  } else {
    return q * (64 * WNB) + lrow;
  }
}

// Compile-time loop: f(std::integral_constant<int, I>) for I in [I0, N).
template <int I0, int N, class Fn>
__device__ __forceinline__ void static_for(Fn&& f) {
  if constexpr (I0 < N) {
    f(std::integral_constant<int, I0>{});
    static_for<I0 + 1, N>(f);
  }
}

// Scheduling groups for an NM-MFMA substep: the NRD fragment reads two after each
// of the first MFMAs (they feed the next substep), then the NWR LDS block writes and
// NVM memory loads spread evenly over the MFMAs from W0 = min(4, NM/2) on, so the
// writes do not queue in the LDS FIFO in front of the reads.  In-order issue means a
// DS instruction stalled on a full FIFO also holds back the MFMAs behind it: with
// reads and writes all front-loaded the K-loop took 8.6% (gate/up) and 5% (down)
// more cycles per step.
template <int NM, int NRD, int NWR, int NVM, int G = 0>
__device__ __forceinline__ void sched_spread() {
  if constexpr (G < NM) {
    constexpr int W0 = NM / 2 < 4 ? NM / 2 : 4;
    constexpr int span = NM - W0, gw = G - W0;
    constexpr int r = 2 * G < NRD ? (NRD - 2 * G < 2 ? NRD - 2 * G : 2) : 0;
    constexpr int w = G < W0 ? 0 : (NWR * (gw + 1)) / span - (NWR * gw) / span;
    constexpr int v = G < W0 ? 0 : (NVM * (gw + 1)) / span - (NVM * gw) / span;
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       // MFMA
    if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);  // DS read
    if constexpr (w > 0) __builtin_amdgcn_sched_group_barrier(0x200, w, 0);  // DS write
    if constexpr (v > 0) __builtin_amdgcn_sched_group_barrier(0x020, v, 0);  // VMEM read
    sched_spread<NM, NRD, NWR, NVM, G + 1>();
  }
}

// Scheduling groups for NM MFMAs with NWR LDS block writes and NVM memory loads spread
// evenly over them (no fragment reads among them).
template <int NM, int NWR, int NVM, int G = 0>
__device__ __forceinline__ void sched_even() {
  if constexpr (G < NM) {
    constexpr int w = (NWR * (G + 1)) / NM - (NWR * G) / NM;
    constexpr int v = (NVM * (G + 1)) / NM - (NVM * G) / NM;
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       // MFMA
    if constexpr (w > 0) __builtin_amdgcn_sched_group_barrier(0x200, w, 0);  // DS write
    if constexpr (v > 0) __builtin_amdgcn_sched_group_barrier(0x020, v, 0);  // VMEM read
    sched_even<NM, NWR, NVM, G + 1>();
  }
}

// Raw buffer resource over [base, base + 4 GiB): loads address it with a 32-bit
// per-lane offset plus a wave-uniform (SGPR) offset, so advancing K costs no VALU.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7fffffff, 0x00020000);
}

// The same over [base, base + bytes): loads past it return 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc_window(const void* base, int64_t bytes) {
  const int n = bytes < 0 ? 0 : (bytes > 0x7fffffffll ? 0x7fffffff : (int)bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, n, 0x00020000);
}

// DUAL products (dx = dg . w1^T + du . w2^T with [dg | du] interleaved per 128 columns, read
// from w1 and w2 (E, d, F) as they are): of four K-steps of 64, the first two are 128
// columns of B, the other two the same columns of B2.
__device__ __forceinline__ bool dual_step_second(int ks) { return ks & 2; }
__device__ __forceinline__ int dual_step_offset(int ks) { return (ks >> 2) * 2 * KB + (ks & 1) * KB; }

struct GemmArgs {
  const uint8_t* A;
  int64_t lda_bytes;
  const float* a_scale;
  const int32_t* row_token;
  const int32_t* row_index;
  const uint8_t* B;
  const uint8_t* B2;  // DUAL tiles: the second weight matrix
  int64_t b_expert_rows;
  int64_t ldb_bytes;
  const float* b_scale;
  int k_bytes;
  uint16_t* C;
  int64_t ldc;
  int n_valid;
  // weight-gradient tiles (OUT_SPLIT): output columns [128, 256) of a tile go to C2
  // and columns [0, 128) to C, both at column nt*128 (the gate and up halves of a
  // w13-ordered tile: the dw1 / dw2 split)
  uint16_t* C2;
  // gate/up tiles: when set, the pre-activation gate and up values are also written
  // (bf16) in the packed column order, row stride 2*ldc: the backward's saved g, u
  uint16_t* gu_out;
  // weight-gradient tiles (OUT_F32): the fp32 accumulators are stored here (row
  // stride ldc) instead of bf16 to C (split-K partial sums)
  float* Cf;
};

// Whether the full tiles of an e4m3 product run in gemm_full_tiles: its pipeline holds two
// K-steps, and its epilogue's buffer stores reach 2 GiB from the tile's first row of C (and of
// gu_out, whose rows are twice as long).  Otherwise every tile runs as narrow ones,
// whose stores take 64-bit addresses.
__host__ __device__ inline bool full_tile_loop(const GemmArgs& g) {
  return g.k_bytes >= 2 * KB && BM * g.ldc * (g.gu_out ? 4 : 2) < (int64_t)1 << 31;
}

// Stores a tile staged in LDS (BM rows of OCPR 16-byte chunks, row stride OSTR bytes)
// to the rows [m0, m_end) of `out` (row stride ld elements, chunk ch at out + 8 ch;
// chunks from column col0 + 8 ch >= n_valid are not stored).  A thread always handles
// the same chunk of every GEMM_THREADS / OCPR-th row, so its addresses advance by a
// fixed stride; LDS reads go out eight at a time ahead of their stores (one read, wait,
// store per iteration serialised the loop on the LDS latency).
template <int OCPR, int OSTR>
__device__ __forceinline__ void store_staged(const uint8_t* lds, int tid, int m0, int m_end, uint16_t* out,
                                             int64_t ld, int col0, int n_valid) {
  constexpr int RPI = GEMM_THREADS / OCPR;  // rows per iteration
  constexpr int NIT = BM / RPI;             // iterations per thread
  constexpr int CH = NIT < 8 ? NIT : 8;
  static_assert(GEMM_THREADS % OCPR == 0 && NIT % CH == 0, "store layout");
  const int ch = tid % OCPR, tr0 = tid / OCPR;
  const bool col_ok = col0 + ch * 8 < n_valid;
  const uint8_t* lp = lds + tr0 * OSTR + ch * 16;
  uint16_t* gp = out + (int64_t)(m0 + tr0) * ld + ch * 8;
  const int rows = m_end - m0 - tr0;  // this thread's rows: tr0 + RPI i < m_end - m0
#pragma unroll
  for (int h = 0; h < NIT; h += CH) {
    i32x4_t v[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) v[u] = *reinterpret_cast<const i32x4_t*>(lp + (h + u) * RPI * OSTR);
#pragma unroll
    for (int u = 0; u < CH; ++u)
      if (col_ok && (h + u) * RPI < rows) *reinterpret_cast<i32x4_t*>(gp + (int64_t)(h + u) * RPI * ld) = v[u];
  }
}

// Output of a weight-gradient tile: bf16 to C; bf16 with the column tile split
// between C and C2 (the gate and up halves of a w13-ordered tile); fp32 to Cf.
constexpr int OUT_BF16 = 0, OUT_SPLIT = 1, OUT_F32 = 2;

// Four values as bf16.
__device__ __forceinline__ i32x2_t pack4_bf16(float a, float b, float c, float d) {
  const uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
  const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{c, d}, bf16x2_t));
  return i32x2_t{(int)lo, (int)hi};
}

// One output tile: rows [m0, min(m0 + 256, m_end)) of expert e against B rows of
// full column tile nt (narrow part q when WNB < 4).
// FP8: A/B bytes are e4m3; a_scale per A row, b_scale per B row (global row index).  Narrow
// tiles only (full ones: gemm_full_tiles), always with NMA = 4.
// GATHER: A is the unpermuted activation matrix and permuted row r is its row
// row_index[row_token[r]] (row_token[r] without row_index): the dispatch gather is
// fused into the A loads.
// RSCALE (bf16 gathered gate/up tiles): a_scale[row_token[r]] scales row r's gate and
// up values before the SiLU (the per-token RMSNorm scale of x: the norm weight is
// folded into the packed w1 / w2 rows, and a per-row scale commutes with the product).
// NMA: the row blocks of this wave that hold rows of the expert.  A wave's 128 rows
// are 4 blocks of 32; a slot's last tile is often partly empty, and its waves then
// run with NMA < 4 (the first NMA blocks), which skips the other blocks' fragment
// reads, MFMAs and epilogue (their accumulators stay 0 and are never stored).  The
// waves of a workgroup may differ in NMA: loads, LDS writes and barriers are the same.
// DUAL: see dual_step_second.
template <bool GATE_UP, bool FP8, bool GATHER, int WNB, bool SAVE_GU = false, bool RSCALE = false, int NMA = 4,
          bool DUAL = false>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, uint8_t* lds, int e, int m0, int m_end, int nt,
                                          int q) {
  static_assert(WNB == 4 || WNB == 2 || WNB == 1, "tile width");
  static_assert(!FP8 || (WNB < 4 && NMA == 4 && !GATHER && !RSCALE && !DUAL), "e4m3 tiles here are narrow");
  // bf16: 16x16x32 MFMAs, 16-row A and B blocks (MA x NBB per wave, NAB of them holding
  // rows); fp8: 32x32x64, 32-row blocks
  constexpr bool M16 = !FP8;
  constexpr int MA = M16 ? 8 : 4;
  constexpr int NAB = M16 ? 2 * NMA : NMA;
  constexpr int NBB = M16 ? 2 * WNB : WNB;
  using Acc = std::conditional_t<M16, f32x4_t, f32x16_t>;
  constexpr int ACCN = M16 ? 4 : 16;
  constexpr int NSUB = KB / 64;  // MFMA K-substeps per pipeline step (bf16: 32 of K, fp8: 64)
  constexpr int BNT = 64 * WNB;                  // B rows of the tile
  constexpr int TBB = BNT * KB;                  // bytes of one B stage tile
  constexpr int BLK_B = BNT * KB / 1024 / 4;     // B load blocks per wave per step
  constexpr int NBLK = BLK_PER_WAVE + BLK_B;     // load blocks per wave per step
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;

  const int64_t brow0 = (int64_t)e * g.b_expert_rows + (int64_t)nt * BN;  // full packed tile
  const __amdgpu_buffer_rsrc_t arsrc = make_rsrc(GATHER ? g.A : g.A + (int64_t)m0 * g.lda_bytes);
  const uint8_t* const bbase = g.B + brow0 * g.ldb_bytes;
  const uint8_t* const b2base = DUAL ? g.B2 + brow0 * g.ldb_bytes : nullptr;
  const __amdgpu_buffer_rsrc_t brsrc = make_rsrc(bbase);
  const int nk = g.k_bytes / KB;
  // LDS stage s: [A tile | B tile]
  auto la_buf = [&](int st) { return lds + st * (TB + TBB); };
  auto lb_buf = [&](int st) { return lds + st * (TB + TBB) + TB; };

  Acc acc[MA][NBB];
#pragma unroll
  for (int i = 0; i < MA; ++i)
#pragma unroll
    for (int j = 0; j < NBB; ++j)
#pragma unroll
      for (int r = 0; r < ACCN; ++r) acc[i][j][r] = 0.0f;
  // fp8 scales of the tile's A rows (thread = row) and B rows (thread = LDS B row),
  // loaded now and put in LDS for the epilogue (rows past the expert's end: 0)
  float sa_v = 0.0f, sb_v = 0.0f;
  if constexpr (FP8) {
    const int row = m0 + tid;
    if (row < m_end) sa_v = g.a_scale[row];
    if (tid < BNT) sb_v = g.b_scale[brow0 + b_packed_row<GATE_UP, WNB>(tid, q)];
  }
  static_assert(!RSCALE || (GATE_UP && GATHER && !FP8 && !SAVE_GU), "row scales are for bf16 gathered gate/up tiles");
  if constexpr (RSCALE) {
    const int row = m0 + tid;
    if (row < m_end) sa_v = g.a_scale[g.row_token[row]];
  }

  // Tile loads: a stage tile is a set of 1 KiB blocks (8 rows of 128 B); wave w loads
  // A blocks [8w, 8w+8) and B blocks [BLK_B w, BLK_B w + BLK_B) into registers and
  // writes them to LDS.  Lane l of a block covers bytes [16l, 16l+16) of it (tile row
  // 8q + l/8, physical chunk l%8) and so loads the logical chunk that swz() maps
  // there: the LDS write of a block is one contiguous, conflict-free 1 KiB.  A rows
  // past the expert's last row read as zeros (their results are never stored).
  const int rsub = lane / CPR, pc = lane % CPR;
  uint32_t a_off[BLK_PER_WAVE], b_off[8];
  const int a_last = m_end - 1 - m0;
  int ra[BLK_PER_WAVE];
#pragma unroll
  for (int qa = 0; qa < BLK_PER_WAVE; ++qa) {
    const int tr = (wave * BLK_PER_WAVE + qa) * RPB + rsub;
    ra[qa] = tr < a_last ? tr : a_last;
  }
  if constexpr (GATHER) {
    // batched: all row_token loads, then all row_index loads (two round trips)
#pragma unroll
    for (int qa = 0; qa < BLK_PER_WAVE; ++qa) ra[qa] = g.row_token[m0 + ra[qa]];
    if (g.row_index) {
#pragma unroll
      for (int qa = 0; qa < BLK_PER_WAVE; ++qa) ra[qa] = g.row_index[ra[qa]];
    }
  }
  // Tile rows past the expert's end load zeros instead: an offset beyond the buffer
  // window's 2 GiB record count makes the hardware return 0 without a memory access
  // (the scalar K offset is not range-checked, the per-lane offset is).  Their results
  // are never stored; zero operands spare the memory traffic and the MFMA power of
  // real data (the expert GEMMs run power-limited).
  constexpr uint32_t A_OOB = 0x80000000u;
#pragma unroll
  for (int qa = 0; qa < BLK_PER_WAVE; ++qa) {
    const int tr = (wave * BLK_PER_WAVE + qa) * RPB + rsub;
    const uint32_t chunk = (uint32_t)(pc ^ ((tr >> 1) & (CPR - 1))) << 4;
    a_off[qa] = tr > a_last ? A_OOB + chunk : (uint32_t)ra[qa] * (uint32_t)g.lda_bytes + chunk;
  }
#pragma unroll
  for (int qb = 0; qb < BLK_B; ++qb) {
    const int tr = (wave * BLK_B + qb) * RPB + rsub;
    const uint32_t chunk = (uint32_t)(pc ^ ((tr >> 1) & (CPR - 1))) << 4;
    b_off[qb] = (uint32_t)b_packed_row<GATE_UP, WNB>(tr, q) * (uint32_t)g.ldb_bytes + chunk;
  }
  i32x4_t stg[16];  // one step of this wave's tile data: A blocks, then B blocks
  // block qq: global -> registers (K-step kt, clamped to the last step)
  auto load_block = [&](int qq, int kt) {
    const int ks = kt < nk ? kt : nk - 1;
    if (qq < BLK_PER_WAVE)
      stg[qq] = __builtin_amdgcn_raw_buffer_load_b128(arsrc, a_off[qq], ks * KB, 0);
    else if constexpr (DUAL)
      stg[qq] = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(dual_step_second(ks) ? b2base : bbase),
                                                      b_off[qq - BLK_PER_WAVE], dual_step_offset(ks), 0);
    else
      stg[qq] = __builtin_amdgcn_raw_buffer_load_b128(brsrc, b_off[qq - BLK_PER_WAVE], ks * KB, 0);
  };
  // block qq: registers -> LDS stage st
  auto write_block = [&](int qq, int st) {
    uint8_t* dst = qq < BLK_PER_WAVE ? la_buf(st) + (wave * BLK_PER_WAVE + qq) * 1024
                                     : lb_buf(st) + (wave * BLK_B + qq - BLK_PER_WAVE) * 1024;
    *reinterpret_cast<i32x4_t*>(dst + lane * 16) = stg[qq];
  };
  Frag<FP8> fa[2][MA], fb[2][NBB];
  const int r16 = lane & 15, lq = lane >> 4;
  // e4m3: all fragments of K-substep i of stage st
  auto rd = [&](int st, int i, Frag<FP8> (&a)[MA], Frag<FP8> (&b)[NBB]) {
    if constexpr (FP8) {
#pragma unroll
      for (int mi = 0; mi < NMA; ++mi) read_frag(la_buf(st), wm * 128 + mi * 32 + lr, i, lh, a[mi]);
#pragma unroll
      for (int j = 0; j < WNB; ++j) read_frag(lb_buf(st), b_lds_row<GATE_UP, WNB>(wn, j, lr), i, lh, b[j]);
    }
  };
  auto mma1 = [&](Acc& c, const Frag<FP8>& b, const Frag<FP8>& a) {
    if constexpr (M16)
      mfma16(c, b, a);
    else
      mfma(c, b, a);
  };
  auto mma = [&](const Frag<FP8> (&a)[MA], const Frag<FP8> (&b)[NBB]) {
#pragma unroll
    for (int mi = 0; mi < NAB; ++mi)
#pragma unroll
      for (int j = 0; j < NBB; ++j) mma1(acc[mi][j], b[j], a[mi]);
  };
  // MFMAs [lo, hi) of a substep (linear index mi * NBB + j)
  auto mma_part = [&](const Frag<FP8> (&a)[MA], const Frag<FP8> (&b)[NBB], auto lo_tag, auto hi_tag) {
    static_for<decltype(lo_tag)::value, decltype(hi_tag)::value>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      mma1(acc[x / NBB][x % NBB], b[x % NBB], a[x / NBB]);
    });
  };

  // Pipeline.  Step kt computes LDS stage kt%2 while the registers hold step kt+1's
  // tile data.  Those blocks are written into stage (kt+1)%2 (which every wave
  // stopped reading at step kt-1's barrier) over the substeps, each block reloaded
  // with step kt+2's data right after its write, so a load has a whole step to land
  // and the LDS write traffic is spread: half of the blocks in each of the two substeps.  In the last substep, after most of
  // its MFMAs, the wave waits for its LDS writes and reads, then one barrier publishes
  // stage kt+1, whose first fragments are read under the last few MFMAs.  Register
  // dependencies give the vmcnt waits; the scheduling groups interleave the LDS and
  // memory operations with the MFMAs, fragment reads first.
  constexpr int RD = 2 * (NAB + NBB);  // e4m3: LDS reads of a substep's fragments
  constexpr int NMS = NAB * NBB;       // MFMAs per substep
  for (int qq = 0; qq < NBLK; ++qq) load_block(qq, 0);
  for (int qq = 0; qq < NBLK; ++qq) write_block(qq, 0);
  for (int qq = 0; qq < NBLK; ++qq) load_block(qq, 1);
  wait_lgkmcnt0();
  barrier_nofence();
  if constexpr (!M16) rd(0, 0, fa[0], fb[0]);

  // bf16 (16x16 blocks): the K loop is emitted in program order, one MFMA at a time,
  // each followed by the LDS reads, block writes or reloads assigned to it and fenced
  // with sched_barrier.  (With scheduling groups the scheduler may take the MFMAs out of
  // order, and the register allocator then stops tying each MFMA's accumulator input to
  // its output: hundreds of accumulator copies per K-step.)  A 16x16x32 MFMA keeps the
  // matrix pipe 16 cycles, about what a 1 KiB LDS block write takes to issue, so the
  // schedule gives each MFMA at most one LDS or memory instruction where it can.
  // Substep i uses B fragment set fb[i] and the one A set fa[0]; MFMAs go row block by
  // row block.  Substep 0 reads substep 1's B fragments into fb[1] and each row block's
  // next A fragment right after that row block's last MFMA (an A ring: no second A set).
  // Substep 1 meets the other waves at the barrier that publishes stage nxt after MFMA
  // GB, then reads that stage's substep-0 fragments (B0, A0, B1, ..., each A after its
  // row block's last MFMA).  The block writes into stage nxt and the reloads of step kt+2
  // go over substep 0 and the part of substep 1 before the barrier, each reload a few
  // MFMAs after the write that frees its registers.
  constexpr bool FULL16 = NMS == 64 && NBB == 8 && NAB == 8 && NBLK == 16;
  constexpr int NR16 = NMS > 0 ? ((NBB + NAB) < NMS - 1 ? NBB + NAB : NMS - 1) : 0;
  constexpr int GB = FULL16 ? 31 : NMS - 1 - NR16;  // substep 1: the barrier follows MFMA GB
  constexpr int H0 = NBLK / 2;                      // block writes in substep 0 (the rest in substep 1)
  auto rdB16 = [&](int st, int i, int j, Frag<FP8>& b) {
    if constexpr (M16) read_frag16(lb_buf(st), b_lds_row<GATE_UP, WNB>(wn, j >> 1, 16 * (j & 1) + r16), i, lq, b);
  };
  auto rdA16 = [&](int st, int i, int mi) {
    if constexpr (M16) read_frag16(la_buf(st), wm * 128 + mi * 16 + r16, i, lq, fa[0][mi]);
  };
  auto sub16 = [&](int kt, auto i_tag, auto last_tag) {
    constexpr int i = decltype(i_tag)::value;
    constexpr bool LAST = decltype(last_tag)::value;
    const int cur = kt & 1, nxt = cur ^ 1;
    constexpr int NW = LAST ? 0 : (i == 0 ? H0 : NBLK - H0), QB = i == 0 ? 0 : H0;
    if constexpr (NMS == 0) {
      // a wave without rows: only its share of the tile loads and the barrier
      if constexpr (NW > 0) {
        static_for<0, NW>([&](auto wc) {
          write_block(QB + decltype(wc)::value, nxt);
          load_block(QB + decltype(wc)::value, kt + 2);
        });
      }
      if constexpr (i == 1 && !LAST) {
        wait_lgkmcnt0();
        barrier_nofence();
      }
      return;
    }
    // MFMA after which block write w / its reload go (w < NW; NW1 keeps the division
    // defined in the instantiations without block writes)
    constexpr int NW1 = NW > 0 ? NW : 1;
    constexpr auto w_at = [](int w) constexpr {
      if (FULL16) return i == 0 ? 16 + 6 * w : 4 * w;
      const int span = i == 0 ? NMS - 2 : GB - 2;
      return span > 0 ? 1 + (w * span) / NW1 : 0;
    };
    constexpr auto l_at = [](int w) constexpr {
      if (FULL16) return i == 0 ? 18 + 6 * w : 4 * w + 2;
      const int span = i == 0 ? NMS - 2 : GB - 2;
      return span > 0 ? 1 + (w * span) / NW1 : 0;
    };
    // substep 0: MFMA after which next-substep read B_j / A_mi goes
    constexpr auto b0_at = [](int j) constexpr { return FULL16 ? 2 * j : (j < NMS ? j : NMS - 1); };
    // substep 1: post-barrier read k (0: B0, 1: A0, 2 ..: B1 .. B_{NBB-1}, then A1 ..)
    constexpr auto post_at = [](int k, int kind, int idx) constexpr {
      const int e0 = GB + 1 + (FULL16 ? 2 * k + 1 : k);
      const int e1 = kind == 1 ? idx * NBB + NBB - 1 : 0;
      const int at = e0 > e1 ? e0 : e1;
      return at < NMS - 1 ? at : NMS - 1;
    };
    static_for<0, NMS>([&](auto gc) {
      constexpr int g = decltype(gc)::value;
      constexpr int mi = g / NBB, j = g % NBB;
      mma1(acc[mi][j], fb[i][j], fa[0][mi]);
      __builtin_amdgcn_sched_barrier(0);
      // block writes, then reloads (substep 1: all before the barrier)
      static_for<0, NW>([&](auto wc) {
        constexpr int w = decltype(wc)::value;
        if constexpr (w_at(w) == g) write_block(QB + w, nxt);
      });
      static_for<0, NW>([&](auto wc) {
        constexpr int w = decltype(wc)::value;
        if constexpr (l_at(w) == g) load_block(QB + w, kt + 2);
      });
      if constexpr (i == 0) {
        static_for<0, NBB>([&](auto jc) {
          constexpr int jj = decltype(jc)::value;
          if constexpr (b0_at(jj) == g) rdB16(cur, 1, jj, fb[1][jj]);
        });
        if constexpr (j == NBB - 1) rdA16(cur, 1, mi);
      } else if constexpr (!LAST) {
        if constexpr (g == GB) {
          wait_lgkmcnt0();
          barrier_nofence();
        }
        static_for<0, NBB + NAB>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          constexpr int kind = k == 0 ? 0 : k == 1 ? 1 : k < NBB + 1 ? 0 : 1;
          constexpr int idx = k == 0 ? 0 : k == 1 ? 0 : k < NBB + 1 ? k - 1 : k - NBB;
          if constexpr (post_at(k, kind, idx) == g) {
            if constexpr (kind == 0)
              rdB16(nxt, 0, idx, fb[0][idx]);
            else
              rdA16(nxt, 0, idx);
          }
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto step16 = [&](int kt, auto last_tag) {
    sub16(kt, std::integral_constant<int, 0>{}, last_tag);
    sub16(kt, std::integral_constant<int, 1>{}, last_tag);
  };
  if constexpr (M16) {
    if constexpr (NMA > 0) {
#pragma unroll
      for (int j = 0; j < NBB; ++j) rdB16(0, 0, j, fb[0][j]);
#pragma unroll
      for (int mi = 0; mi < NAB; ++mi) rdA16(0, 0, mi);
    }
  }
  auto step = [&](int kt, auto last_tag) {
    if constexpr (M16) return step16(kt, last_tag);
    constexpr bool LAST = decltype(last_tag)::value;
    const int cur = kt & 1, nxt = cur ^ 1;
    static_for<0, NSUB>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr int bi = i & 1;
      // blocks [q0, q1) are written and reloaded in this substep: half in each, the last
      // substep's before its barrier (all in substep 0 crowded the LDS queue with that
      // substep's fragment reads: 3% slower)
      constexpr int q0 = i * NBLK / NSUB, q1 = (i + 1) * NBLK / NSUB;
      constexpr int nq = LAST ? 0 : q1 - q0;
      constexpr bool RDN = i + 1 < NSUB || !LAST;
      // next substep's fragments first: they are on the MFMA critical path
      if constexpr (i + 1 < NSUB) {
        rd(cur, i + 1, fa[bi ^ 1], fb[bi ^ 1]);
      } else if constexpr (!LAST) {
        // last substep: its share of the block writes and most of its MFMAs go out before
        // the wait and the barrier that publish the next stage (the MFMAs read registers
        // only), so the MFMA pipe is busy while the waves meet; the next stage's first
        // fragment reads then issue two per MFMA under the remaining NA.  (Barrier first:
        // each step lost the pipe for the wait on the writes plus the barrier.)
        constexpr int NA = (RD + 1) / 2 < NMS ? (RD + 1) / 2 : NMS;
        if constexpr (nq > 0) {
          static_for<q0, q1>([&](auto qc) { write_block(decltype(qc)::value, nxt); });
          static_for<q0, q1>([&](auto qc) { load_block(decltype(qc)::value, kt + 2); });
        }
        if constexpr (NMS - NA > 0) {
          mma_part(fa[bi], fb[bi], std::integral_constant<int, 0>{}, std::integral_constant<int, NMS - NA>{});
          sched_even<NMS - NA, nq, nq>();
        }
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkmcnt0();
        barrier_nofence();
        rd(nxt, 0, fa[bi ^ 1], fb[bi ^ 1]);
        if constexpr (NA > 0) {
          mma_part(fa[bi], fb[bi], std::integral_constant<int, NMS - NA>{}, std::integral_constant<int, NMS>{});
          sched_spread<NA, RD, 0, 0>();
        }
        __builtin_amdgcn_sched_barrier(0);
        return;
      }
      if constexpr (nq > 0) {
        static_for<q0, q1>([&](auto qc) { write_block(decltype(qc)::value, nxt); });
        static_for<q0, q1>([&](auto qc) { load_block(decltype(qc)::value, kt + 2); });
      }
      mma(fa[bi], fb[bi]);
      sched_spread<NMS, (RDN ? RD : 0), nq, nq>();
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  for (int kt = 0; kt + 1 < nk; ++kt) step(kt, std::false_type{});
  step(nk - 1, std::true_type{});

  // ---- epilogue.  The MFMAs take the B fragment as their first operand, so block
  // (mi, j) accumulates the transposed product: acc[mi][j][4c+t] is A row mi*32 + lr
  // against B row 8c + 4lh + t of B block j, i.e. output row wm*128 + mi*32 + lr and
  // four consecutive output columns per c.  A lane packs each such run to 8 bytes of
  // bf16 in registers and writes it to an LDS tile (rows padded by 16 bytes), which
  // then goes out with 16-byte stores along rows.
  static_assert(!SAVE_GU || GATE_UP, "g/u saving is for gate/up tiles");
  static_assert(!(SAVE_GU && FP8 && M16), "fp8 tiles use 32x32 blocks");
  constexpr int NC = GATE_UP ? 32 * WNB : 64 * WNB;  // output columns of the tile
  // output column blocks per wave, and 4-column runs per block and lane: a gate/up
  // WNB = 1 block holds its gate values in runs c = 0, 1 and the up values of the same
  // columns in runs c + 2
  constexpr bool GU1 = GATE_UP && WNB == 1;
  constexpr int NJ = GU1 ? 1 : GATE_UP ? WNB / 2 : WNB;
  constexpr int NCR = GU1 ? 2 : 4;
  constexpr int OSTR = NC * 2 + 16;                  // LDS row stride (bytes)
  float* const sa_l = reinterpret_cast<float*>(lds + SCALE_LDS);
  float* const sb_l = sa_l + BM;
  if constexpr (FP8) {
    sa_l[tid] = sa_v;
    if (tid < BNT) sb_l[tid] = sb_v;
  }
  if constexpr (RSCALE) sa_l[tid] = sa_v;
  __syncthreads();
  // The scales go to registers first: the B-row scales of the lane's 16 B rows of each
  // block once, the A-row scale of each row block before its results.  Read from LDS
  // per output element, they were re-read after every staging write (the compiler
  // cannot tell the two LDS areas apart).
  float sbr[WNB][16];
#pragma unroll
  for (int j = 0; j < WNB; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      sbr[j][r] = FP8 ? sb_l[b_lds_row<GATE_UP, WNB>(wn, j, 8 * (r >> 2) + 4 * lh + (r & 3))] : 1.0f;
  float sar = 1.0f;
  // e4m3: output r of block (mi, jo), descaled
  auto result = [&](int mi, int r, int jo) -> float {
    if (GATE_UP) {
      constexpr int UJ = GU1 ? 0 : WNB / 2, UR = GU1 ? 8 : 0;  // up value: block jo + UJ, run + UR/4
      const float gg = acc[mi][jo][r] * (sar * sbr[jo][r]);
      const float u = acc[mi][jo + UJ][r + UR] * (sar * sbr[jo + UJ][r + UR]);
      return silu_fast_f32(gg) * u;
    } else {
      return acc[mi][jo][r] * (sar * sbr[jo][r]);
    }
  };
  if constexpr (M16) {
    // 16x16 blocks: acc[mi][j][t] is output row wm*128 + mi*16 + l%16 against B row
    // 4 (l/16) + t of 16-row B block j: one run of four output columns per block (gate/up:
    // gate block jo, up block jo + NBB/2, same columns)
    constexpr int NJ16 = GATE_UP ? NBB / 2 : NBB;
    uint8_t* const wb16 = lds + (wm * 128 + r16) * OSTR + (wn * (NC / 2) + 4 * lq) * 2;
#pragma unroll
    for (int mi = 0; mi < NAB; ++mi) {
      if constexpr (RSCALE) sar = sa_l[wm * 128 + mi * 16 + r16];
#pragma unroll
      for (int jo = 0; jo < NJ16; ++jo) {
        float v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if constexpr (GATE_UP) {
            float gg = acc[mi][jo][t], u = acc[mi][jo + NBB / 2][t];
            if constexpr (RSCALE) {
              gg *= sar;
              u *= sar;
            }
            v[t] = silu_fast_f32(gg) * u;
          } else {
            v[t] = acc[mi][jo][t];
          }
        }
        *reinterpret_cast<i32x2_t*>(wb16 + mi * 16 * OSTR + jo * 32) = pack4_bf16(v[0], v[1], v[2], v[3]);
      }
    }
  } else {
    // lane's row of block 0 and its first column (c = 0) of output column block 0
    uint8_t* const wbase = lds + (wm * 128 + lr) * OSTR + (wn * (NC / 2) + 4 * lh) * 2;
#pragma unroll
    for (int mi = 0; mi < NMA; ++mi) {
      sar = sa_l[wm * 128 + mi * 32 + lr];
#pragma unroll
      for (int jo = 0; jo < NJ; ++jo)
#pragma unroll
        for (int c = 0; c < NCR; ++c)
          *reinterpret_cast<i32x2_t*>(wbase + mi * 32 * OSTR + (jo * 32 + 8 * c) * 2) =
              pack4_bf16(result(mi, 4 * c, jo), result(mi, 4 * c + 1, jo), result(mi, 4 * c + 2, jo),
                    result(mi, 4 * c + 3, jo));
    }
  }
  __syncthreads();
  constexpr int OCPR = NC * 2 / 16;  // 16-byte chunks per output row
  const int col0 = (GATE_UP ? nt * 128 : nt * 256) + q * NC;
  store_staged<OCPR, OSTR>(lds, tid, m0, m_end, g.C + col0, g.ldc, col0, g.n_valid);

  // training forward: the pre-activation gate and up values of the tile, bf16, in the
  // packed column order (row stride 2*ldc), for the SwiGLU backward (fp8: descaled by
  // the row and column scales, the values the SwiGLU of the epilogue took)
  if constexpr (SAVE_GU) {
    constexpr int NC2 = 64 * WNB;
    constexpr int OSTR2 = NC2 * 2 + 16;
    __syncthreads();
    if constexpr (M16) {
      uint8_t* const wb2 = lds + (wm * 128 + r16) * OSTR2 + 4 * lq * 2;
#pragma unroll
      for (int mi = 0; mi < NAB; ++mi)
#pragma unroll
        for (int j = 0; j < NBB; ++j) {
          const int col = b_lds_row<true, WNB>(wn, j >> 1, 16 * (j & 1));
          *reinterpret_cast<i32x2_t*>(wb2 + mi * 16 * OSTR2 + col * 2) =
              pack4_bf16(acc[mi][j][0], acc[mi][j][1], acc[mi][j][2], acc[mi][j][3]);
        }
    } else {
      uint8_t* const wb2 = lds + (wm * 128 + lr) * OSTR2 + 4 * lh * 2;
#pragma unroll
      for (int mi = 0; mi < NMA; ++mi) {
        sar = sa_l[wm * 128 + mi * 32 + lr];
#pragma unroll
        for (int j = 0; j < WNB; ++j) {
          const int col = b_lds_row<true, WNB>(wn, j, 0);
          auto gv = [&](int r) { return acc[mi][j][r] * (sar * sbr[j][r]); };
#pragma unroll
          for (int c = 0; c < 4; ++c)
            *reinterpret_cast<i32x2_t*>(wb2 + mi * 32 * OSTR2 + (col + 8 * c) * 2) =
                pack4_bf16(gv(4 * c), gv(4 * c + 1), gv(4 * c + 2), gv(4 * c + 3));
        }
      }
    }
    __syncthreads();
    constexpr int OCPR2 = NC2 * 2 / 16;
    // chunk ch of a staged row lands at packed column b_packed_row(8 ch): contiguous
    // within each 8-column chunk, so the per-thread base column is that of its chunk
    const int ch2 = tid % OCPR2;
    const int gcol2 = nt * 256 + b_packed_row<true, WNB>(ch2 * 8, q);
    store_staged<OCPR2, OSTR2>(lds, tid, m0, m_end, g.gu_out + gcol2 - ch2 * 8, 2 * g.ldc, 0, 1 << 30);
  }
}

// The half waves of a 32x32 block hold runs of four output columns 8c + 4 (lane / 32) (two
// dwords of bf16): from runs x = c and y = c + 1 a lane gets the eight consecutive columns
// of run c + lane / 32, one 16-byte store.
__device__ __forceinline__ i32x4_t merge32(i32x2_t x, i32x2_t y) {
  const auto a = __builtin_amdgcn_permlane32_swap((unsigned)x[0], (unsigned)y[0], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap((unsigned)x[1], (unsigned)y[1], false, false);
  return i32x4_t{(int)a[0], (int)b[0], (int)a[1], (int)b[1]};
}
// LDS of the full-tile loop behind its stages: the experts' slot table (lo, hi, inclusive
// slot count of each) and two sets of A-row and B-row scales.
constexpr int FT_SLOTS = NST * 2 * TB;
constexpr int FT_SCALE = FT_SLOTS + 1024;
constexpr int FT_LDS = FT_SCALE + 2 * 2 * BM * 4;
static_assert(FT_LDS <= GEMM_LDS, "LDS of the full-tile loop");

// The full 256 x 256 tiles of a workgroup of an e4m3 product: tiles L = blockIdx.x, + n_cu,
// .. < n_full, in one continuous K pipeline.  The last two K-steps of a tile load the next
// tile's first two (its scales were looked up at the start of the tile), so the next tile
// starts with its first stage in LDS and its second step in flight, and the epilogue
// stores straight from registers.  One workgroup fills a CU (128 KiB of stages, 512
// registers), so whatever runs between two tiles leaves its matrix cores idle, and an
// e4m3 tile has half the K-steps of a bf16 one: 12288 rows over 16 experts, d 2048, F
// 2816, gate/up + down 216 -> 197 us against one workgroup per tile.  (bf16 tiles the same way: 1045
// -> 1025 us at 16384 tokens, eleven rounds, but 2% slower at one to three rounds; they
// stay one workgroup per tile.)  For products with full_tile_loop().
// NMA (4, 2, 1 or 0, per tile and wave): the wave's 32-row blocks that hold rows of the
// expert; the others' fragment reads, MFMAs and stores are skipped.  The waves of a
// workgroup may differ in NMA: loads, LDS writes and barriers are the same.
// a_scale per A row, b_scale per B row (global row index).
template <bool GATE_UP, bool SAVE_GU>
__device__ __forceinline__ void gemm_full_tiles(const GemmArgs& g, uint8_t* lds, const SlotTable& st, int E,
                                                int n_tiles, int n_cu, int base, int n_full) {
  constexpr int MA = 4, NBB = 4;              // 32-row A and B blocks of a wave
  constexpr int NSUB = KB / 64;               // MFMA K-substeps per step (64 of K)
  constexpr int NBLK = 2 * BLK_PER_WAVE;      // load blocks per wave per step: A, then B
  static_assert(!SAVE_GU || GATE_UP, "g/u saving is for gate/up tiles");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  const int nk = g.k_bytes / KB;
  int L = blockIdx.x;
  if (L >= n_full) return;

  // slot table to LDS (every wave holds the same: wave 0 writes it; read after a barrier)
  int* const slot_l = reinterpret_cast<int*>(lds + FT_SLOTS);
  float* const sc_l = reinterpret_cast<float*>(lds + FT_SCALE);
  {
    int incl = st.ns;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (lane >= o) incl += u;
    }
    if (wave == 0) {
      slot_l[lane] = st.lo;
      slot_l[64 + lane] = st.hi;
      slot_l[128 + lane] = incl;
    }
  }
  __syncthreads();
  // A lane number that the compiler takes for new: what is computed from it stays inside
  // the tile loop.  (Hoisted out of it, the addresses of the lookups and of the epilogue
  // take the registers that the K loop needs and end up in scratch memory.)
  auto fresh = [](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  struct Tile {
    int e, m0, m_end, nt;
  };
  auto decode = [&](int l) -> Tile {
    const int t = (l < base && base % (NXCD * SB_TILES) == 0) ? xcd_tile(l) : l;
    int slot;
    Tile r;
    dense_tile(t, st.n_slots, n_tiles, slot, r.nt);
    const int fl = fresh(lane);
    const int lo = slot_l[fl], hi = slot_l[64 + fl], incl = slot_l[128 + fl];
    r.e = __builtin_ctzll(__ballot(slot < incl));  // slot < n_slots: some lane holds it
    const int before = r.e > 0 ? __builtin_amdgcn_readlane(incl, r.e - 1) : 0;
    r.m0 = __builtin_amdgcn_readlane(lo, r.e) + (slot - before) * BM;
    r.m_end = __builtin_amdgcn_readlane(hi, r.e);
    return r;
  };

  // Tile loads: a stage tile is a set of 1 KiB blocks (8 rows of 128 B); wave w loads
  // blocks [8w, 8w + 8) of A and of B into registers and writes them to LDS.  Lane l of a
  // block covers bytes [16l, 16l+16) of it (tile row 8q + l/8, physical chunk l%8) and so
  // loads the logical chunk that swz() maps there: the LDS write of a block is one
  // contiguous, conflict-free 1 KiB.
  constexpr uint32_t OOB = 0x80000000u;  // an offset past every buffer window
  const int rsub = lane / CPR, pc = lane % CPR;
  uint32_t a_off[BLK_PER_WAVE], b_off[BLK_PER_WAVE];
#pragma unroll
  for (int q = 0; q < BLK_PER_WAVE; ++q) {
    const int tr = (wave * BLK_PER_WAVE + q) * RPB + rsub;
    const uint32_t chunk = (uint32_t)(pc ^ ((tr >> 1) & (CPR - 1))) << 4;
    a_off[q] = (uint32_t)tr * (uint32_t)g.lda_bytes + chunk;
    b_off[q] = (uint32_t)tr * (uint32_t)g.ldb_bytes + chunk;
  }
  __amdgpu_buffer_rsrc_t arsrc, brsrc;
  int koff = 0;
  // points the loads at tile t (any = false: at nothing).  The A window ends at the
  // expert's last row; loads past a window return zeros without a memory access (the
  // scalar K offset is not range-checked, the per-lane offset is): the rows past the end
  // are never stored, and zero operands spare traffic and MFMA power.
  auto aim = [&](const Tile& t, bool any) {
    const int rows = t.m_end - t.m0;
    brsrc = make_rsrc_window(g.B + ((int64_t)t.e * g.b_expert_rows + (int64_t)t.nt * BN) * g.ldb_bytes,
                             any ? 0x7fffffff : 0);
    arsrc = make_rsrc_window(g.A + (int64_t)t.m0 * g.lda_bytes, any ? (int64_t)rows * g.lda_bytes : 0);
  };
  // thread tid looks up the scales of tile row tid and of B row tid
  auto look_scales = [&](const Tile& t, float& sa, float& sb) {
    const int ft = fresh(tid), r = t.m0 + ft;
    sa = r < t.m_end ? g.a_scale[r] : 0.0f;
    sb = g.b_scale[(int64_t)t.e * g.b_expert_rows + (int64_t)t.nt * BN + ft];
  };
  auto put_scales = [&](int set, float sa, float sb) {
    const int ft = fresh(tid);
    sc_l[set * 2 * BM + ft] = sa;
    sc_l[set * 2 * BM + BM + ft] = sb;
  };

  i32x4_t stg[NBLK];  // one step of this wave's tile data
  auto load_block = [&](int qq) {
    if (qq < BLK_PER_WAVE)
      stg[qq] = __builtin_amdgcn_raw_buffer_load_b128(arsrc, a_off[qq], koff, 0);
    else
      stg[qq] = __builtin_amdgcn_raw_buffer_load_b128(brsrc, b_off[qq - BLK_PER_WAVE], koff, 0);
  };
  auto la_buf = [&](int s) { return lds + s * 2 * TB; };
  auto lb_buf = [&](int s) { return lds + s * 2 * TB + TB; };
  auto write_block = [&](int qq, int s) {
    uint8_t* dst = qq < BLK_PER_WAVE ? la_buf(s) + (wave * BLK_PER_WAVE + qq) * 1024
                                     : lb_buf(s) + (wave * BLK_PER_WAVE + qq - BLK_PER_WAVE) * 1024;
    *reinterpret_cast<i32x4_t*>(dst + lane * 16) = stg[qq];
  };

  f32x16_t acc[MA][NBB];
  Frag<true> fa[2][MA], fb[2][NBB];
  auto rd = [&](int s, int i, auto nma_tag, Frag<true> (&a)[MA], Frag<true> (&b)[NBB]) {
    constexpr int NMA = decltype(nma_tag)::value;
    if constexpr (NMA > 0) {
#pragma unroll
      for (int mi = 0; mi < NMA; ++mi) read_frag(la_buf(s), wm * 128 + mi * 32 + lr, i, lh, a[mi]);
#pragma unroll
      for (int j = 0; j < NBB; ++j) read_frag(lb_buf(s), b_lds_row<GATE_UP, 4>(wn, j, lr), i, lh, b[j]);
    }
  };

  // One K-step on stage cur while the registers hold the following step's data: those
  // blocks are written into stage cur ^ 1 (which every wave stopped reading at the
  // previous step's barrier) over the substeps, each reloaded at koff right after its
  // write, so a load has a whole step to land and the LDS write traffic is spread.  In the
  // last substep the wave waits for its LDS writes and reads, then one barrier publishes
  // stage cur ^ 1, whose first fragments are read under the remaining MFMAs.  Register
  // dependencies give the vmcnt waits.
  // Half of the block writes and reloads go in each of the two substeps,
  // fragments double buffered, interleaved by scheduling groups; in the last substep the
  // writes and most MFMAs go out before the wait and the barrier (the MFMAs read registers
  // only), so the MFMA pipe is busy while the waves meet.
  auto step = [&](int cur, auto nma_tag) {
    constexpr int NMA = decltype(nma_tag)::value;
    constexpr int RD = NMA > 0 ? 2 * (NMA + NBB) : 0;  // LDS reads of a substep's fragments
    constexpr int NMS = NMA * NBB;
    const int nxt = cur ^ 1;
    auto mma_part = [&](const Frag<true> (&a)[MA], const Frag<true> (&b)[NBB], auto lo_tag, auto hi_tag) {
      static_for<decltype(lo_tag)::value, decltype(hi_tag)::value>([&](auto xc) {
        constexpr int x = decltype(xc)::value;
        mfma(acc[x / NBB][x % NBB], b[x % NBB], a[x / NBB]);
      });
    };
    static_for<0, NSUB>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr int bi = i & 1;
      constexpr int q0 = i * NBLK / NSUB, q1 = (i + 1) * NBLK / NSUB;
      constexpr int nq = q1 - q0;
      if constexpr (i + 1 < NSUB) rd(cur, i + 1, nma_tag, fa[bi ^ 1], fb[bi ^ 1]);
      static_for<q0, q1>([&](auto qc) { write_block(decltype(qc)::value, nxt); });
      static_for<q0, q1>([&](auto qc) { load_block(decltype(qc)::value); });
      if constexpr (i + 1 < NSUB) {
        mma_part(fa[bi], fb[bi], std::integral_constant<int, 0>{}, std::integral_constant<int, NMS>{});
        sched_spread<NMS, RD, nq, nq>();
        __builtin_amdgcn_sched_barrier(0);
      } else {
        constexpr int NA = (RD + 1) / 2 < NMS ? (RD + 1) / 2 : NMS;
        if constexpr (NMS - NA > 0) {
          mma_part(fa[bi], fb[bi], std::integral_constant<int, 0>{}, std::integral_constant<int, NMS - NA>{});
          sched_even<NMS - NA, nq, nq>();
        }
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkmcnt0();
        barrier_nofence();
        rd(nxt, 0, nma_tag, fa[bi ^ 1], fb[bi ^ 1]);
        if constexpr (NA > 0) {
          mma_part(fa[bi], fb[bi], std::integral_constant<int, NMS - NA>{}, std::integral_constant<int, NMS>{});
          sched_spread<NA, RD, 0, 0>();
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };

  // Epilogue: a lane's runs of four consecutive output columns are packed to bf16, merged
  // in pairs to 16 bytes across lanes and stored by buffer stores whose offset of a row or
  // column that does not exist is out of the buffer's range (dropped by the hardware).
  auto epilogue = [&](const Tile& t, int set, auto nma_tag) {
    constexpr int NMA = decltype(nma_tag)::value;
    if constexpr (NMA > 0) {
      const int fl = fresh(lane), lr = fl & 31, lh = fl >> 5;
      const float* const sa_l = sc_l + set * 2 * BM;
      const float* const sb_l = sa_l + BM;
      const __amdgpu_buffer_rsrc_t crsrc = make_rsrc(g.C + (int64_t)t.m0 * g.ldc);
      const __amdgpu_buffer_rsrc_t grsrc = make_rsrc(SAVE_GU ? g.gu_out + (int64_t)t.m0 * 2 * g.ldc : g.C);
      const int rows = t.m_end - t.m0;
      const uint32_t ldc2 = (uint32_t)g.ldc * 2u;
      const int col0 = (GATE_UP ? t.nt * 128 : t.nt * 256) + wn * (GATE_UP ? 64 : 128);
      constexpr int NJ = GATE_UP ? NBB / 2 : NBB;
#pragma unroll
      for (int mi = 0; mi < NMA; ++mi) {
        const int row = wm * 128 + mi * 32 + lr;
        const float sar = sa_l[row];
        const uint32_t roff = row < rows ? (uint32_t)row * ldc2 : OOB;
        const uint32_t goff = row < rows ? (uint32_t)row * 2u * ldc2 : OOB;
#pragma unroll
        for (int jo = 0; jo < NJ; ++jo) {
#pragma unroll
          for (int cp = 0; cp < 4; cp += 2) {
            i32x2_t v[2], vg[2], vu[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int c = cp + h;
              const f32x4_t sb =
                  *reinterpret_cast<const f32x4_t*>(sb_l + b_lds_row<GATE_UP, 4>(wn, jo, 8 * c + 4 * lh));
              float f[4], gv[4], uv[4];
              f32x4_t su = sb;
              if constexpr (GATE_UP)
                su = *reinterpret_cast<const f32x4_t*>(sb_l + b_lds_row<GATE_UP, 4>(wn, jo + NBB / 2, 8 * c + 4 * lh));
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                gv[q] = acc[mi][jo][4 * c + q] * (sar * sb[q]);
                if constexpr (GATE_UP) {
                  uv[q] = acc[mi][jo + NBB / 2][4 * c + q] * (sar * su[q]);
                  f[q] = silu_fast_f32(gv[q]) * uv[q];
                } else {
                  f[q] = gv[q];
                }
              }
              v[h] = pack4_bf16(f[0], f[1], f[2], f[3]);
              if constexpr (SAVE_GU) {
                vg[h] = pack4_bf16(gv[0], gv[1], gv[2], gv[3]);
                vu[h] = pack4_bf16(uv[0], uv[1], uv[2], uv[3]);
              }
            }
            const int lcol = 8 * (cp + lh);
            const int col = col0 + jo * 32 + lcol;
            const uint32_t off = col < g.n_valid ? roff + 2u * (uint32_t)col : OOB;
            __builtin_amdgcn_raw_buffer_store_b128(merge32(v[0], v[1]), crsrc, off, 0, 0);
            if constexpr (SAVE_GU) {
              const uint32_t cg = (uint32_t)(t.nt * 256 + b_lds_row<true, 4>(wn, jo, 0) + lcol);
              const uint32_t cu = (uint32_t)(t.nt * 256 + b_lds_row<true, 4>(wn, jo + NBB / 2, 0) + lcol);
              __builtin_amdgcn_raw_buffer_store_b128(merge32(vg[0], vg[1]), grsrc, goff + 2u * cg, 0, 0);
              __builtin_amdgcn_raw_buffer_store_b128(merge32(vu[0], vu[1]), grsrc, goff + 2u * cu, 0, 0);
            }
          }
        }
      }
    }
  };

  // the first tile: looked up and started with nothing in flight (step 0 to stage 0, step 1
  // in registers)
  Tile cur = decode(L);
  {
    float sa, sb;
    look_scales(cur, sa, sb);
    put_scales(0, sa, sb);
    aim(cur, true);
    koff = 0;
#pragma unroll
    for (int qq = 0; qq < NBLK; ++qq) load_block(qq);
#pragma unroll
    for (int qq = 0; qq < NBLK; ++qq) write_block(qq, 0);
    koff = KB;
#pragma unroll
    for (int qq = 0; qq < NBLK; ++qq) load_block(qq);
    wait_lgkmcnt0();
    barrier_nofence();
  }
  int par = 0;  // stage of the tile's step 0
  int set = 0;  // scale set of the tile
  bool more;
  do {
    more = L + n_cu < n_full;
    if (more) L += n_cu;
    const Tile nx = decode(L);
    auto body = [&](auto nma_tag) {
      constexpr int NMA = decltype(nma_tag)::value;
      if constexpr (NMA > 0) {
        rd(par, 0, nma_tag, fa[0], fb[0]);
#pragma unroll
        for (int i = 0; i < NMA; ++i)
#pragma unroll
          for (int j = 0; j < NBB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
      }
      float sa, sb;
      look_scales(nx, sa, sb);
#pragma unroll 1
      for (int kt = 0; kt < nk; ++kt) {
        koff = (kt + 2) * KB;
        if (kt >= nk - 2) {
          // the last two steps load the next tile's first two
          koff = (kt + 2 - nk) * KB;
          if (kt == nk - 2) {
            // (with two steps nothing else keeps this write behind the other waves' reads of
            // the set in the previous tile's epilogue)
            if (nk == 2) barrier_nofence();
            put_scales(set ^ 1, sa, sb);
            aim(nx, more);
          }
        }
        step((par + kt) & 1, nma_tag);
      }
      // every accumulator leaves the loop in AGPRs, and the epilogue stays out of its last
      // step (else the allocator spills in the loop)
#pragma unroll
      for (int i = 0; i < NMA; ++i)
#pragma unroll
        for (int j = 0; j < NBB; ++j) asm volatile("" : "+a"(acc[i][j]));
      __builtin_amdgcn_sched_barrier(0);
      epilogue(cur, set, nma_tag);
    };
    // row blocks of this wave holding rows (wave-uniform): 4 (more than 64 rows), 2, 1, 0
    const int wrows = cur.m_end - cur.m0 - wm * 128;
    if (wrows > 64)
      body(std::integral_constant<int, 4>{});
    else if (wrows > 32)
      body(std::integral_constant<int, 2>{});
    else if (wrows > 0)
      body(std::integral_constant<int, 1>{});
    else
      body(std::integral_constant<int, 0>{});
    cur = nx;
    par = (par + nk) & 1;
    set ^= 1;
  } while (more);
}

// Work of workgroup blockIdx.x.  The tiles (slot, column tile) are numbered densely
// (dense_tile); with n_cu workgroups resident at a time, the first R = N/n_cu full
// rounds take one tile per workgroup in the XCD-aware order.  The N - R n_cu tiles
// left would occupy few compute units for a whole tile time, so when they fit
// (split > 1: at most n_cu / split of them) each is split into `split` narrow tiles
// of 1/split of its columns (the full K), which all run at once.  A narrow tile
// computes every output element with the same MFMA sequence as the full tile, so
// the results are identical.  split = 1 keeps the tail tiles whole.
// e4m3 products with full_tile_loop(): the full rounds (and whole tail tiles) go to
// gemm_full_tiles on the first n_cu workgroups, the narrow tiles to the ones after them
// (without it: all tiles in halves or quarters).
template <bool GATE_UP, bool FP8, bool GATHER, bool SAVE_GU = false, bool RSCALE = false, bool DUAL = false>
__global__ __launch_bounds__(GEMM_THREADS, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void grouped_gemm_kernel(
    GemmArgs g, const int32_t* __restrict__ offsets, int E, int n_tiles, int n_cu) {
  static_assert(!(GATHER && FP8), "the fp8 path reads rows quantised by the dispatch");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[GEMM_LDS];
  const SlotTable st = load_slots(offsets, E);
  const int n_all = st.n_slots * n_tiles;
  const int rounds = n_all / n_cu, base = rounds * n_cu, n_rest = n_all - base;
  int split = 1;
  if (n_rest > 0) {
    if (4 * n_rest <= n_cu)
      split = 4;
    else if (2 * n_rest <= n_cu)
      split = 2;
  }
  const int L = blockIdx.x;
  if constexpr (FP8) {
    // without the loop every tile is narrow, in quarters where all of them then fit at once
    const bool halves = !full_tile_loop(g);
    if (halves) split = 4 * n_all <= n_cu ? 4 : 2;
    // the narrow tiles wait behind n_cu workgroups only where those have tiles of their own
    // (4 experts, d 256, F 352, 1024 rows: gate/up + down 13.8 us behind 256 workgroups
    // without one, 12.8 from the first on), and a single K-step takes quarters where all fit
    // at once (16 experts, d 128, F 256, 128 rows: 14.5 us in halves, 12.1)
    const int first = halves ? 0 : base;  // first narrow tile
    const bool looped = !halves && (split == 1 || base > 0);
    if (looped && L < n_cu) {
      gemm_full_tiles<GATE_UP, SAVE_GU>(g, lds, st, E, n_tiles, n_cu, base, split == 1 ? n_all : base);
      return;
    }
    const int u = looped ? L - n_cu : L;
    if (split == 1 || u >= (n_all - first) * split) return;
    int slot, nt, e, m0, m_end;
    dense_tile(first + u / split, st.n_slots, n_tiles, slot, nt);
    find_slot(st, E, slot, e, m0, m_end);
    if (split == 2)
      gemm_tile<GATE_UP, true, false, 2, SAVE_GU, false>(g, lds, e, m0, m_end, nt, u % split);
    else
      gemm_tile<GATE_UP, true, false, 1, SAVE_GU, false>(g, lds, e, m0, m_end, nt, u % split);
    return;
  } else {
    int t, q = 0;
    if (L < base) {
      t = (base % (NXCD * SB_TILES)) == 0 ? xcd_tile(L) : L;
    } else if (split == 1) {
      if (L >= n_all) return;
      t = L;
    } else {
      const int u = L - base;
      if (u >= n_rest * split) return;
      t = base + u / split;
      q = u % split;
    }
    int slot, nt, e, m0, m_end;
    dense_tile(t, st.n_slots, n_tiles, slot, nt);
    find_slot(st, E, slot, e, m0, m_end);
    if (L < base || split == 1) {
      // row blocks of this wave holding rows (wave-uniform): 4 (more than 64 rows), 2, 1, 0
      const int wrows = m_end - m0 - (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >> 1) * 128;
      if (wrows > 64)
        gemm_tile<GATE_UP, FP8, GATHER, 4, SAVE_GU, RSCALE, 4, DUAL>(g, lds, e, m0, m_end, nt, 0);
      else if (wrows > 32)
        gemm_tile<GATE_UP, FP8, GATHER, 4, SAVE_GU, RSCALE, 2, DUAL>(g, lds, e, m0, m_end, nt, 0);
      else if (wrows > 0)
        gemm_tile<GATE_UP, FP8, GATHER, 4, SAVE_GU, RSCALE, 1, DUAL>(g, lds, e, m0, m_end, nt, 0);
      else
        gemm_tile<GATE_UP, FP8, GATHER, 4, SAVE_GU, RSCALE, 0, DUAL>(g, lds, e, m0, m_end, nt, 0);
    } else if (split == 2)
      gemm_tile<GATE_UP, FP8, GATHER, 2, SAVE_GU, RSCALE, 4, DUAL>(g, lds, e, m0, m_end, nt, q);
    else
      gemm_tile<GATE_UP, FP8, GATHER, 1, SAVE_GU, RSCALE, 4, DUAL>(g, lds, e, m0, m_end, nt, q);
  }
}

// One grouped product to launch: the kernel's arguments, grid and stream.  The kernel's
// variants are compiled in separate files (each takes a minute); these launch them.
struct GemmLaunch {
  GemmArgs g;
  const int32_t* offsets;
  int E, n_tiles, n_cu;
  unsigned blocks;
  hipStream_t s;
};
template <bool GATE_UP, bool FP8, bool GATHER, bool SAVE_GU = false, bool RSCALE = false, bool DUAL = false>
void launch_variant(const GemmLaunch& l) {
  hipLaunchKernelGGL((grouped_gemm_kernel<GATE_UP, FP8, GATHER, SAVE_GU, RSCALE, DUAL>), dim3(l.blocks),
                     dim3(GEMM_THREADS), 0, l.s, l.g, l.offsets, l.E, l.n_tiles, l.n_cu);
}
void launch_gate_up_rows(const GemmLaunch& l);                    // bf16, gathered rows (RSCALE with a_scale)
void launch_gate_up_rows_gu(const GemmLaunch& l);                 // the same, saving the gate / up values
void launch_permuted(const GemmLaunch& l, bool gate_up);          // bf16, permuted rows
void launch_dual(const GemmLaunch& l);                            // the same, no gate/up, weights from B and B2
void launch_fp8(const GemmLaunch& l, bool gate_up, bool save_gu); // e4m3, permuted rows
// bf16, few rows per expert (kmoe_gemm_small.hip): slots of SMALL_ROWS rows, n_tiles column
// tiles of small_cols() output columns
constexpr int SMALL_ROWS = 32;
inline int small_cols(bool gate_up) { return gate_up ? 16 : 32; }
void launch_small_rows(const GemmLaunch& l, bool gate_up);

}  // namespace kmoe_tiles
