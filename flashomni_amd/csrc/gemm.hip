// GEMM-Q and GEMM-O (with reduction) for gfx950: MFMA tile GEMMs that skip work according to the
// bit-packed (token-block, head) flags.
//
//   GEMM-Q  y[b, iy-tile, ix-tile] = x[b, iy-tile, :] . w[ix-tile, :]^T + bias   for flagged tiles;
//           the other tiles are never touched (reference: gemm/w16a16/gemm.cuh:50-58, 83-92).
//   GEMM-O  y[b, iy-tile, :] = init + sum_{selected heads h} x[:, h-slice] . w[:, h-slice]^T
//           where unselected head slices are never loaded
//           (reference: gemm/w16a16/gemm_reduction.cuh:77-95, 126-160).
//
// Tiling.  The skip flags have a 128 x 128 granularity ("unit"), but a CU can pull only ~50-60 B/clk
// from L2 while its matrix cores eat a 128 x 128 x 64 step in ~500 clocks, so small workgroup tiles
// starve.  A workgroup (4 wavefronts, one per SIMD, 512 registers each) therefore computes a *quad*:
// two token blocks x two column blocks that share their operand tiles (four 128 x 64 tiles feed four
// units).  A wavefront owns one unit: 128 x 128 accumulators (256 registers, kept in the accumulator
// half of the register file), sixteen MFMAs per eight 128-bit operand reads.  (With eight wavefronts
// of 64 x 128 the same loop spent a third more LDS reads per MFMA and ran 25 % slower.)  A list
// kernel packs the flagged units of every (16-token-block window, column pair) cell into work items:
// rows flagged in both columns pair up into full quads; rows flagged in one column go three at a time
// into *column strips* (three token blocks x that column block: three X tiles and one W tile, three
// wavefronts busy), what is left pairs up or is merged; a mask says which units of an item exist
// (the wavefront of a missing unit only moves data).  With four fifths of the units flagged at
// random (the 14B-video configuration) that fills 86 % of the wavefront slots against 81 % with
// quads alone, from the same operand tiles, and the launch is 2 % shorter.  (Measured and dropped:
// items dealt by row pair over the whole width, full quads for the columns both token blocks have and
// strips of one token block x three column blocks for the rest: 91 % of the slots, but a strip's
// three columns lie far apart and few concurrent items share its W tiles, 9.4 GB fetched per launch
// against 6.8 GB, and the launch was 1.3 % shorter.  Either way the time per round of work items
// rises with the fill.)  GEMM-Q with is_full computes every unit: no list then, the
// kernel derives its quads from the shape.  GEMM-O, whose token blocks differ in length, runs as strips
// (gemm_strip_kernel).
//
// Data path.  Operands are staged in slabs of 64 k: a tile row is then 128 B, one whole memory line.
// A wavefront fetches its sixteen 8-row pieces of a slab with buffer loads (a resource descriptor
// per tile in scalar registers, 32-bit lane offsets, the k offset as the scalar offset: no vector
// address arithmetic; rows past M read as zeros through the descriptor's range check) into staging registers one slab ahead, and writes them to LDS (two slab buffers) a slab
// later; loads, LDS writes and operand reads are spread evenly between the MFMAs (per sixteen MFMAs:
// eight reads, four writes, four loads), so the memory path sees an even stream and nothing queues
// behind a burst.  (Direct global -> LDS copies need no registers but can only be issued once a
// buffer is free, i.e. in a burst after the barrier: the issue stalls of that burst, 100-150 clocks
// per copy and wavefront, cost a quarter of the loop.)  One barrier per slab.  Rows are XOR-swizzled
// instead of padded: row r keeps logical 16-byte chunk c at position c ^ ((r >> 1) & 7), applied to
// the LDS write address; the 128-bit operand reads of 16 consecutive rows then cover all 64 banks.
// A k range that is not a multiple of 64 (K = 32 mod 64) ends in a slab
// that reaches 32 back into its neighbour; that half of its X operand is cleared on the way to LDS
// (a separate instantiation, so that the common case carries no masking).
//
// The product is formed transposed (A operand = W rows, B operand = X rows): in the 32 x 32
// accumulator layout a lane owns one output row and runs of 4 consecutive columns.  Stored (or the
// init matrix read) from that layout, a wavefront instruction is 64 scattered 8-byte pieces, so the
// epilogue turns each wavefront's block through its own quarter of the (by then free) slab buffers,
// 32 rows at a time in fp32, into a layout where 32 consecutive lanes cover one row; there the bias
// vector or the cached partial is added in fp32 and the result is rounded once and stored through a
// buffer descriptor that ends with the matrix (no per-row tests).  The first slab of the next work
// item is requested before the epilogue, so that its latency hides behind the stores.
//
// Launches of few units and launches whose quads would leave CUs idle run a workgroup per unit or per strip instead
// (gemm_deep_kernel, gemm_unit_kernel, gemm_packed_kernel, gemm_strip_kernel, and the rules in launch_o and launch_q).
//
// Work order.  Workgroups are persistent (one per CU).  The quad list is ordered by token window,
// then column pair, then row pair, and XCD x (= blockIdx % 8) owns the x-th contiguous eighth of it.
// The ~32 workgroups of an XCD therefore work at the same time on one token window and four
// neighbouring column pairs (16 + 8 operand tiles for 32 quads), whose tiles they share through
// that XCD's L2; work items of equal length keep them in step in k, which is what makes the tiles
// hit (measured at the Wan size: 6.8 GB fetched per launch against 28 GB of operand loads).
#include "fo_common.h"
#include "fo_device.h"
#include "fo_flags.h"

#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

constexpr int kThreads = 256;
constexpr int kTile = 128;  // unit edge = granularity of the skip flags
constexpr int kBK = 64;                            // k range of one LDS slab
constexpr int kRowBytes = kBK * 2;                 // one LDS row: 64 elements = one 128-byte memory line, 8 chunks of 16 B
constexpr int kUnitBytes = kTile * kRowBytes;      // one 128-row operand tile: 16 KB
constexpr int kStageBytes = 4 * kUnitBytes;        // X0, X1, W0, W1
constexpr int kStages = 2;
constexpr int kSmemBytes = kStages * kStageBytes;  // 128 KB
constexpr int kUnitSmemBytes = kStages * 2 * kUnitBytes;  // workgroup per unit: 64 KB, two workgroups per CU
constexpr int kDeepThreads = 768;  // ... one per CU, or a strip of two units: W column blocks take four wavefronts each, the rest copy
constexpr int deep_ring(int W) { return W == 1 ? 5 : 3; }
constexpr int deep_smem_bytes(int W) { return deep_ring(W) * (1 + W) * kUnitBytes; }  // 160, 144 KB
constexpr int kUnitWindow = 8;  // ... token blocks per scheduling window
constexpr int kZeroFirst = 1 << 18, kZeroSecond = 1 << 19;  // slab entry: half of the slab does not count
constexpr int kMaxHeads = 256;
constexpr int kMaxSteps = 2048;  // GEMM-O: k steps of one work item (K <= 65536)
constexpr int kXcds = 8;
constexpr int kListThreads = 1024;
constexpr int kInlineCells = 256;  // up to this many cells the GEMM-Q kernel lists its quads itself
constexpr int kWindow = 16;   // token blocks per scheduling window
constexpr int kQuadInts = 8;  // b, r0, r1, c0, c1, valid mask, r2 (column strips), pad
constexpr int kColStrip = 0x20;        // in the valid mask: the item is a column strip (three token blocks x one column block)
constexpr int kColStripSecond = 0x40;  // ... of the cell's second column

template <typename T>
struct Types;
template <>
struct Types<__bf16> {
  using x8 = bf16x8;
  using x4 = bf16x4;
  static __device__ __forceinline__ f32x16 mfma(x8 a, x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(x8 a, x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Types<_Float16> {
  using x8 = f16x8;
  using x4 = f16x4;
  static __device__ __forceinline__ f32x16 mfma(x8 a, x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(x8 a, x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

struct GemmParams {
  const void* x;     // [B, M, K]
  const void* w;     // [N, K]
  const void* bias;  // [N] or [B, M, N] or null
  void* y;           // [B, M, N]
  const uint8_t* sparse_info;
  const int32_t* sparse_info_indptr;
  const int32_t* quads;  // kQuadInts per quad, queue by queue; null: the kernel lists them itself (inline_cells), or every
                         // unit is computed and the quads are enumerated arithmetically (is_full)
  const int32_t* qoff;   // qoff[0..8] queue boundaries inside `quads`
  int32_t n_row_tiles, n_col_tiles, n_cp;  // geometry for the arithmetic enumeration
  int32_t strip_cols;    // strips: column groups of XCDs
  int32_t strip_sorted;  // strips: token blocks with the most selected heads first
  int32_t num_cu;        // strips of flagged units: up to as many have a CU each
  int32_t* judgement;    // GEMM-Q: the word in which quads leave to the strips behind them whether they ran, or null
  int32_t n_win;         // windows of 16 token blocks per batch
  int32_t inline_cells;  // > 0: GEMM-Q builds its quad list itself from the flags of this many cells
  int32_t batch, m, n, k;
  int32_t sparse_q_size, num_heads, head_dim, num_text_tokens;
  int32_t flag;       // GEMM-Q: is_full.  GEMM-O: is_for_cached
  int32_t bias_kind;  // FO_BIAS_*
  int32_t bias_f32;   // matrix bias is fp32
  int32_t y_f32;      // output is fp32
  // GEMM-Q with fused quantisation: e4m3fn bytes [B, M, N] and one scale per (head, token block),
  // y_scale[head * scale_row_len + b * n_row_tiles + token block]; y may then be null
  uint8_t* y8;
  uint8_t* y8_lo;  // optional second term: the residual result / scale - y8, rounded to e4m3 again
  float* y_scale;
  int32_t scale_row_len;
};

__device__ __forceinline__ bool flag_bit(const uint8_t* info, uint32_t bit) {
  return (info[bit >> 3] >> (bit & 7)) & 1;
}

// ---------------------------------------------------------------------------------------------
// Quad list.  A cell = (batch, window of 16 token blocks, column pair); cells are ordered batch,
// window, column pair.  One workgroup counts the quads of every cell (flagged-row masks of its two
// columns), scans the counts, emits every cell's quads at its offset, and cuts the list into eight
// contiguous, equally long queues.  (Up to kInlineCells cells the GEMM-Q kernel does the same itself.)
// ---------------------------------------------------------------------------------------------
struct ListGeom {
  int32_t batch, n_row_tiles, n_col_tiles, n_win, n_cp;  // windows per batch, column pairs
};

__device__ __forceinline__ void cell_masks(const ListGeom& gm, int cell,
                                           const uint8_t* __restrict__ sparse_info,
                                           const int32_t* __restrict__ sparse_info_indptr,
                                           int32_t sparse_q_size, int32_t num_heads, int32_t head_dim,
                                           int32_t num_text_tokens, int* b_out, int* row0_out,
                                           int* cp_out, uint32_t* m0, uint32_t* m1) {
  const int cp = cell % gm.n_cp;
  const int t = cell / gm.n_cp;
  const int w = t % gm.n_win, b = t / gm.n_win;
  *b_out = b;
  *row0_out = w * kWindow;
  *cp_out = cp;
  const int rows = min(kWindow, gm.n_row_tiles - w * kWindow);
  const uint32_t all = (1u << rows) - 1u;
  const bool has1 = 2 * cp + 1 < gm.n_col_tiles;
  const uint8_t* info = sparse_info + sparse_info_indptr[b];
  // All flag bytes of the cell are requested before the first is looked at (rows past the end repeat
  // the last one): one memory latency for the cell instead of one per row.
  const uint32_t head0 = static_cast<uint32_t>(2 * cp * kTile) / head_dim;
  const uint32_t head1 = has1 ? static_cast<uint32_t>((2 * cp + 1) * kTile) / head_dim : head0;
  const bool unit_blocks = sparse_q_size == kTile;  // flag blocks = token blocks: no division per row
  const uint32_t text_blocks = static_cast<uint32_t>(num_text_tokens) / kTile;
  uint32_t bit0[kWindow], bit1[kWindow];
  uint8_t byte0[kWindow], byte1[kWindow];
#pragma unroll
  for (int r = 0; r < kWindow; ++r) {
    const int row = w * kWindow + min(r, rows - 1);
    const uint32_t blk = unit_blocks ? text_blocks + static_cast<uint32_t>(row)
                                     : static_cast<uint32_t>(num_text_tokens + row * kTile) / sparse_q_size;
    bit0[r] = blk * num_heads + head0;
    bit1[r] = blk * num_heads + head1;
    byte0[r] = info[bit0[r] >> 3];
    byte1[r] = info[bit1[r] >> 3];
  }
  uint32_t a0 = 0, a1 = 0;
#pragma unroll
  for (int r = 0; r < kWindow; ++r) {
    a0 |= ((byte0[r] >> (bit0[r] & 7)) & 1u) << r;
    a1 |= ((byte1[r] >> (bit1[r] & 7)) & 1u) << r;
  }
  *m0 = a0 & all;
  *m1 = has1 ? a1 & all : 0u;
}

__device__ __forceinline__ int pop_lowest(uint32_t* m) {
  const int r = __ffs(*m) - 1;
  *m &= *m - 1;
  return r;
}

// Packs a cell's flagged units into work items and calls f(r0, r1, valid, r2) for each; r1 < 0 = no
// second row.  Quads: valid bits 1 = (r0,c0), 2 = (r0,c1), 4 = (r1,c0), 8 = (r1,c1).  Column strips:
// valid = kColStrip | 7 (| kColStripSecond for the cell's second column), rows r0, r1, r2 of that column.
template <typename F>
__device__ __forceinline__ void for_each_quad(uint32_t m0, uint32_t m1, F&& f) {
  uint32_t both = m0 & m1, only0 = m0 & ~m1, only1 = m1 & ~m0;
  while (__popc(both) >= 2) {
    const int r0 = pop_lowest(&both), r1 = pop_lowest(&both);
    f(r0, r1, 0xF, 0);
  }
  // rows flagged in one column only: three at a time into a column strip (three X tiles, one W tile)
  while (__popc(only0) >= 3) {
    const int r0 = pop_lowest(&only0), r1 = pop_lowest(&only0), r2 = pop_lowest(&only0);
    f(r0, r1, kColStrip | 0x7, r2);
  }
  while (__popc(only1) >= 3) {
    const int r0 = pop_lowest(&only1), r1 = pop_lowest(&only1), r2 = pop_lowest(&only1);
    f(r0, r1, kColStrip | kColStripSecond | 0x7, r2);
  }
  while (__popc(only0) >= 2) {
    const int r0 = pop_lowest(&only0), r1 = pop_lowest(&only0);
    f(r0, r1, 0x5, 0);
  }
  while (__popc(only1) >= 2) {
    const int r0 = pop_lowest(&only1), r1 = pop_lowest(&only1);
    f(r0, r1, 0xA, 0);
  }
  // at most one row left in each class: merge them two by two
  if (both) {
    const int r0 = pop_lowest(&both);
    if (only0) {
      f(r0, pop_lowest(&only0), 0x3 | 0x4, 0);
    } else if (only1) {
      f(r0, pop_lowest(&only1), 0x3 | 0x8, 0);
    } else {
      f(r0, -1, 0x3, 0);
    }
  }
  if (only0 && only1) {
    const int r0 = pop_lowest(&only0);
    f(r0, pop_lowest(&only1), 0x1 | 0x8, 0);
  } else if (only0) {
    f(pop_lowest(&only0), -1, 0x1, 0);
  } else if (only1) {
    f(pop_lowest(&only1), -1, 0x2, 0);
  }
}

// The same for work items of at most two units that share a tile (`pairs`, see gemm_kernel): two rows of a
// column, or both columns of a row, or one unit.
template <typename F>
__device__ __forceinline__ void for_each_pair(uint32_t m0, uint32_t m1, F&& f) {
  while (__popc(m0) >= 2) {
    const int r0 = pop_lowest(&m0), r1 = pop_lowest(&m0);
    f(r0, r1, 0x5, 0);
  }
  while (__popc(m1) >= 2) {
    const int r0 = pop_lowest(&m1), r1 = pop_lowest(&m1);
    f(r0, r1, 0xA, 0);
  }
  if (m0 && m0 == m1) {
    f(pop_lowest(&m0), -1, 0x3, 0);
  } else {
    if (m0) f(pop_lowest(&m0), -1, 0x1, 0);
    if (m1) f(pop_lowest(&m1), -1, 0x2, 0);
  }
}
// how many that are: of an odd number of rows the last one is left over
__device__ __forceinline__ int count_pairs(uint32_t m0, uint32_t m1) {
  const int n0 = __popc(m0), n1 = __popc(m1);
  const bool together = (n0 & n1 & 1) && __clz(m0) == __clz(m1);
  return (n0 + 1) / 2 + (n1 + 1) / 2 - (together ? 1 : 0);
}

struct ListArgs {
  const uint8_t* sparse_info;
  const int32_t* sparse_info_indptr;
  int32_t sparse_q_size, num_heads, head_dim, num_text_tokens;
};

__global__ void __launch_bounds__(kListThreads) gemm_quads_kernel(ListArgs a, ListGeom gm,
                                                                  int32_t* __restrict__ quads,
                                                                  int32_t* __restrict__ qoff) {
  __shared__ int32_t s_cnt[kListThreads / 64];
  const int tid = threadIdx.x;
  const int n_cells = gm.batch * gm.n_win * gm.n_cp;
  int b, row0, cp;
  uint32_t m0, m1;
  // every thread owns a contiguous run of cells: quad counts, then a block-wide scan
  const int per = (n_cells + kListThreads - 1) / kListThreads;
  const int lo = min(tid * per, n_cells), hi = min(lo + per, n_cells);
  int32_t my_cnt = 0;
  for (int cell = lo; cell < hi; ++cell) {
    cell_masks(gm, cell, a.sparse_info, a.sparse_info_indptr, a.sparse_q_size, a.num_heads,
               a.head_dim, a.num_text_tokens, &b, &row0, &cp, &m0, &m1);
    for_each_quad(m0, m1, [&](int, int, int, int) { ++my_cnt; });
  }
  // inclusive scan of the per-thread counts: inside a wavefront by lane shifts, then over the
  // sixteen wavefront totals
  const int lane = tid & 63, wave = tid >> 6;
  int32_t incl = my_cnt;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t up = __shfl_up(incl, d, 64);
    if (lane >= d) incl += up;
  }
  if (lane == 63) s_cnt[wave] = incl;
  __syncthreads();
  int32_t wave_base = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kListThreads / 64; ++w) {
    const int32_t t = s_cnt[w];
    if (w < wave) wave_base += t;
    total += t;
  }
  const int32_t my_incl = wave_base + incl;
  if (tid <= kXcds) qoff[tid] = static_cast<int32_t>(static_cast<int64_t>(total) * tid / kXcds);
  int32_t q = my_incl - my_cnt;
  for (int cell = lo; cell < hi; ++cell) {
    if (per > 1)  // with one cell per thread the masks of the counting pass are still at hand
      cell_masks(gm, cell, a.sparse_info, a.sparse_info_indptr, a.sparse_q_size, a.num_heads,
                 a.head_dim, a.num_text_tokens, &b, &row0, &cp, &m0, &m1);
    for_each_quad(m0, m1, [&](int r0, int r1, int valid, int r2) {
      int32_t* e = quads + kQuadInts * static_cast<int64_t>(q);
      e[0] = b;
      e[1] = row0 + r0;
      e[2] = row0 + (r1 < 0 ? r0 : r1);
      if (valid & kColStrip) {
        e[3] = e[4] = (valid & kColStripSecond) ? 2 * cp + 1 : 2 * cp;
      } else {
        e[3] = (valid & 0x5) ? 2 * cp : 2 * cp + 1;
        e[4] = (valid & 0xA) ? 2 * cp + 1 : 2 * cp;
      }
      e[5] = valid;
      e[6] = row0 + r2;
      ++q;
    });
  }
}

// ---------------------------------------------------------------------------------------------
// GEMM-Q as quads.  kQuant: with fused quantisation (an epilogue with register needs of its own).
// ---------------------------------------------------------------------------------------------
template <typename T, bool kHalf, bool kQuant>
__global__ void __launch_bounds__(kThreads) gemm_kernel(const GemmParams p) {
  using TT = Types<T>;
  using x8 = typename TT::x8;
  using x4 = typename TT::x4;
  constexpr int NT = 4, MT = 4;  // wavefront tile = one unit: 128 columns (W rows) x 128 token rows (X rows)
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // GEMM-Q listing its own quads (short launches: saves the list kernel's launch): quad count
  // prefix and flagged-row masks of every cell, and the entry picked for the current work item
  __shared__ int32_t s_cell_pref[kInlineCells + 1];
  __shared__ uint32_t s_cell_mask[2 * kInlineCells];
  __shared__ int32_t s_cell_wave[kThreads / 64];
  __shared__ int32_t s_entry[8];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);  // wavefront index = unit of the quad, kept scalar
  const int l32 = lane & 31, g = lane >> 5;
  const int wr = wv >> 1, wc = wv & 1;  // token block, column block

  const T* __restrict__ xg = static_cast<const T*>(p.x);
  const T* __restrict__ wg = static_cast<const T*>(p.w);

  // Load assignment: a slab is 64 pieces of 8 rows x 128 B (whole memory lines), 16 per wavefront:
  // pieces 0..7 = rows 64*(wv%2) + 8*j.. of X tile wv/2, pieces 8..15 = the same rows of W tile wv/2.
  // Lane i fetches 16-byte chunk i%8 of row i/8 of its piece and writes it to LDS at chunk position
  // (i%8) ^ ((row >> 1) & 7) = (i%8) ^ ((4*(j%2) + (i >> 4)) & 7).
  const int ld_row = 64 * (wv & 1) + (lane >> 3), ld_chunk = lane & 7;
  int wr_off[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    wr_off[par] = (lane >> 3) * kRowBytes + ((ld_chunk ^ ((4 * par + (lane >> 4)) & 7)) << 4);
  // lanes that hold the first / the second half of a slab's k range
  const unsigned mask_first = ld_chunk < 4 ? 0xFFFFFFFFu : 0u;
  // operand reads: row = tile row base + l32 (bases are multiples of 32), logical chunk 2*s + g of substep s
  const int rd_x = (g ^ ((l32 >> 1) & 7)) << 4;

  const int xcd = blockIdx.x & (kXcds - 1), slot = blockIdx.x >> 3;
  const int per_xcd = gridDim.x >> 3;  // host launches a multiple of 8 workgroups
  // dense enumeration (same order as the list kernel's): per batch, windows of 16 token blocks
  // (8 row pairs; the last window may be shorter), column pairs inside a window, row pairs inside
  // a column pair
  const int full_w = p.n_row_tiles / kWindow, last_rows = p.n_row_tiles % kWindow;
  constexpr int per_win = kWindow / 2;  // work items per window and column pair
  const int last_q = (last_rows + 1) / 2;
  const int quads_per_batch = (full_w * per_win + last_q) * p.n_cp;
  int q_lo, q_len;
  const bool inline_list = p.inline_cells > 0;
  // Few flagged units (GEMM-Q that lists its own work): a quad would keep one CU busy for four units' time
  // while others idle.  If items of at most two units are no more than the workgroups, the list is made of
  // those, and two wavefronts share a unit: each takes two of a slab's four substeps (half of k), and the
  // halves are added through LDS at the end.  Measured with K = 3072 (us, quads -> pairs): 16 k tokens x 24
  // heads with one unit in ten flagged 60 -> 45, 4.6 k tokens with a quarter flagged 60 -> 43.  The error
  // against 64-bit sums is the same (bf16 1.66e-3, fp16 2.08e-4: the rounding of the result).
  constexpr bool kPairs = !kQuant;
  bool pairs = false;
  if (inline_list) {
    // thread = cell: masks, quad count, workgroup-wide inclusive scan of the counts
    ListGeom gm;
    gm.batch = p.batch;
    gm.n_row_tiles = p.n_row_tiles;
    gm.n_col_tiles = p.n_col_tiles;
    gm.n_win = p.n_win;
    gm.n_cp = p.n_cp;
    int32_t cnt = 0;
    if (tid < p.inline_cells) {
      int b, row0, cp;
      uint32_t m0, m1;
      cell_masks(gm, tid, p.sparse_info, p.sparse_info_indptr, p.sparse_q_size, p.num_heads,
                 p.head_dim, p.num_text_tokens, &b, &row0, &cp, &m0, &m1);
      for_each_quad(m0, m1, [&](int, int, int, int) { ++cnt; });
      if constexpr (kPairs) {  // (both counts in one scan: at most 16 per cell and kInlineCells cells)
        cnt += count_pairs(m0, m1) << 16;
      }
      s_cell_mask[2 * tid] = m0;
      s_cell_mask[2 * tid + 1] = m1;
    }
    int32_t incl = cnt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t up = __shfl_up(incl, d, 64);
      if (lane >= d) incl += up;
    }
    if (lane == 63) s_cell_wave[wv] = incl;
    __syncthreads();
    int32_t base = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) {
      const int32_t t = s_cell_wave[w];
      if (w < wv) base += t;
      total += t;
    }
    incl += base;
    if constexpr (kPairs) {
      pairs = (total >> 16) <= static_cast<int>(gridDim.x);
      total = pairs ? total >> 16 : total & 0xFFFF;
      incl = pairs ? incl >> 16 : incl & 0xFFFF;
      if (p.judgement != nullptr) {  // (a launch of strips follows, which reads whose turn it is: launch_q)
        int units = tid < p.inline_cells ? __popc(s_cell_mask[2 * tid]) + __popc(s_cell_mask[2 * tid + 1]) : 0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) units += __shfl_xor(units, off, 64);
        if (lane == 0) s_entry[wv] = units;
        __syncthreads();
        units = s_entry[0] + s_entry[1] + s_entry[2] + s_entry[3];
        // (strips: half of a token block's two groups of columns will hold an odd number)
        const int cus = gridDim.x, strips = (units + p.batch * p.n_row_tiles) / 2;
        const bool mine = !pairs && total <= cus && strips > cus;
        if (blockIdx.x == 0 && tid == 0) *p.judgement = mine;
        if (!mine) return;
      }
    }
    if (tid < kInlineCells) s_cell_pref[tid + 1] = incl;
    if (tid == 0) s_cell_pref[0] = 0;
    q_lo = static_cast<int>(static_cast<int64_t>(total) * xcd / kXcds);
    q_len = static_cast<int>(static_cast<int64_t>(total) * (xcd + 1) / kXcds) - q_lo;
    __syncthreads();
  } else if (p.quads) {
    q_lo = p.qoff[xcd];
    q_len = p.qoff[xcd + 1] - q_lo;
  } else {
    const int64_t total = static_cast<int64_t>(quads_per_batch) * p.batch;
    q_lo = static_cast<int>(total * xcd / kXcds);
    q_len = static_cast<int>(total * (xcd + 1) / kXcds) - q_lo;
  }

  // ---- work items ----
  // A work item = a quad: four operand tiles per slab (X r0, X r1, W c0, W c1), wavefront = unit,
  // 128 x 128 each; or a column strip (X r0, X r1, W c0, X r2).  (Another shape was measured and dropped: quads with two units that share a
  // tile, computed by two wavefronts per unit at 64 x 128 each from three tiles.  Its slab takes as
  // long as a full one (nine LDS transfers per eight MFMAs saturate a wavefront's LDS path), and work
  // items of unequal length let the workgroups of an XCD drift apart in k, which costs the L2 hits on
  // the tiles they share.)
  constexpr int P = 16;      // pieces per wavefront and slab: rows 32*wv + 8*jj.. (jj = 0..3) of every tile
  constexpr int PS = P / 4;  // pieces per substep
  // valid & kColStrip (GEMM-Q with flags): the item is a column strip, three token blocks r[0], r[1],
  // r2 x one column block c[0] (tiles: X r[0], X r[1], W c[0], X r2; wavefronts 0..2 own the units).
  struct Item {
    int bz, valid, r[2], c[2], r2;
  };
  // (called by all threads together: the listing form hands the entry over through LDS)
  auto decode_item = [&](int work) -> Item {
    int bz, valid, r[2], c[2], r2 = 0;
    if (inline_list) {
      // the thread whose cell holds quad q_lo + work walks the cell's quads up to it
      const int q = q_lo + work;
      if (tid < p.inline_cells && s_cell_pref[tid] <= q && q < s_cell_pref[tid + 1]) {
        const int cp = tid % p.n_cp, t = tid / p.n_cp;
        const int w = t % p.n_win, b = t / p.n_win;
        int k = q - s_cell_pref[tid];
        auto entry = [&](int r0, int r1, int v, int r2) {
          if (k == 0) {
            s_entry[0] = b;
            s_entry[1] = w * kWindow + r0;
            s_entry[2] = w * kWindow + (r1 < 0 ? r0 : r1);
            if (v & kColStrip) {
              s_entry[3] = s_entry[4] = (v & kColStripSecond) ? 2 * cp + 1 : 2 * cp;
            } else {
              s_entry[3] = (v & 0x5) ? 2 * cp : 2 * cp + 1;
              s_entry[4] = (v & 0xA) ? 2 * cp + 1 : 2 * cp;
            }
            s_entry[5] = v;
            s_entry[6] = w * kWindow + r2;
          }
          --k;
        };
        if (kPairs && pairs) {
          for_each_pair(s_cell_mask[2 * tid], s_cell_mask[2 * tid + 1], entry);
        } else {
          for_each_quad(s_cell_mask[2 * tid], s_cell_mask[2 * tid + 1], entry);
        }
      }
      __syncthreads();
      bz = s_entry[0];
      r[0] = s_entry[1];
      r[1] = s_entry[2];
      c[0] = s_entry[3];
      c[1] = s_entry[4];
      valid = s_entry[5];
      r2 = s_entry[6];
    } else if (p.quads) {
      const int32_t* e = p.quads + kQuadInts * static_cast<int64_t>(q_lo + work);
      bz = e[0];
      r[0] = e[1];
      r[1] = e[2];
      c[0] = e[3];
      c[1] = e[4];
      valid = e[5];
      r2 = e[6];
    } else {
      const int q = q_lo + work;
      bz = q / quads_per_batch;
      int rem = q - bz * quads_per_batch;
      int w, cp, i, rows;
      if (rem < full_w * p.n_cp * per_win) {
        const int cell = rem / per_win;
        i = rem - cell * per_win;
        w = cell / p.n_cp;
        cp = cell - w * p.n_cp;
        rows = kWindow;
      } else {
        rem -= full_w * p.n_cp * per_win;
        cp = rem / last_q;
        i = rem - cp * last_q;
        w = full_w;
        rows = last_rows;
      }
      const bool has_r1 = 2 * i + 1 < rows, has_c1 = 2 * cp + 1 < p.n_col_tiles;
      r[0] = w * kWindow + 2 * i;
      r[1] = has_r1 ? r[0] + 1 : r[0];
      c[0] = 2 * cp;
      c[1] = has_c1 ? c[0] + 1 : c[0];
      valid = 0x1 | (has_c1 ? 0x2 : 0) | (has_r1 ? 0x4 : 0) | (has_r1 && has_c1 ? 0x8 : 0);
    }
    Item it;
    it.bz = __builtin_amdgcn_readfirstlane(bz);
    it.valid = __builtin_amdgcn_readfirstlane(valid);
    it.r2 = __builtin_amdgcn_readfirstlane(r2);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      it.r[u] = __builtin_amdgcn_readfirstlane(r[u]);
      it.c[u] = __builtin_amdgcn_readfirstlane(c[u]);
    }
    return it;
  };
  const int n_iter = (p.k + kBK - 1) / kBK;
  // k offset of step it (steps past the end repeat the last one)
  auto step_entry = [&](int it) -> int {
    // (K % 64 == 32: the last slab reaches 32 back and counts for its second half only)
    const int i = it < n_iter ? it : n_iter - 1;
    return (i + 1) * kBK <= p.k ? i * kBK : (p.k - kBK) | kZeroFirst;
  };
  // ---- operand tiles: buffer resource descriptors in scalar registers ----
  // The X descriptors end with the matrix, so rows past M read as zeros.
  const __amdgpu_buffer_rsrc_t rsrc_none = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(xg), 0, 0, 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc[4] = {rsrc_none, rsrc_none, rsrc_none, rsrc_none};
  auto make_rsrc = [&](const Item& item) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int rows_left = min(p.m - item.r[u] * kTile, kTile);  // >= 1
      rsrc[u] = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<T*>(xg + (static_cast<int64_t>(item.bz) * p.m + static_cast<int64_t>(item.r[u]) * kTile) * p.k), 0,
          rows_left * p.k * 2, 0x00020000);
      rsrc[2 + u] = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<T*>(wg + static_cast<int64_t>(item.c[u]) * kTile * p.k), 0, kTile * p.k * 2, 0x00020000);
    }
    if (item.valid & kColStrip) {  // a column strip's fourth tile is its third X tile
      const int rows_left = min(p.m - item.r2 * kTile, kTile);
      rsrc[3] = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<T*>(xg + (static_cast<int64_t>(item.bz) * p.m + static_cast<int64_t>(item.r2) * kTile) * p.k), 0,
          rows_left * p.k * 2, 0x00020000);
    }
  };
  int ld_off[4];
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) ld_off[jj] = (32 * wv + 8 * jj + (lane >> 3)) * p.k * 2 + ld_chunk * 16;
  // Staging registers: piece j of a slab waits here between its global load and its LDS write.
  u32x4 stg[P];
  auto gload = [&](int j, int entry) {
    stg[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc[j >> 2], ld_off[j & 3], (entry & 0xFFFF) * 2, 0);
  };
  // kHalf: only the second half of a slab that reaches into its neighbour counts; the first half of the X
  // pieces is cleared on the way to LDS
  auto keep_of = [&](int entry) -> unsigned {
    return (entry & kZeroFirst) ? ~mask_first : 0xFFFFFFFFu;
  };
  auto lwrite = [&](int j, int stage, unsigned keep) {
    const int t = j >> 2;
    uint8_t* dst = smem + stage * kStageBytes + t * kUnitBytes + (32 * wv + 8 * (j & 3)) * kRowBytes + wr_off[j & 1];
    u32x4 v = stg[j];
    if constexpr (kHalf) {
      if (t != 2) v &= keep;  // (every tile that can hold X; a W tile cleared along with its X tile changes nothing)
    }
    *reinterpret_cast<u32x4*>(dst) = v;
  };

  if constexpr (kPairs) {
    if (pairs) {
      // One item of at most two units (no more items than workgroups), two wavefronts each.
      if (slot >= q_len) return;
      const Item item = decode_item(slot);
      // Three tiles at most: X r0, X r1, W of a column pair; X, W c0, W c1 of a row's two units; X, none, W.
      // (What the loop waits for is the vector memory path: a CU takes ~37 bytes per clock through it, and
      // loads that fetch nothing hold it up as well: with four tiles, one or two of them empty, 51 and 47 us.
      // Two slabs in flight in staging registers, against the latency of a tile's first touch, do not fit
      // the registers beside 256 accumulators: 757 spilled.)
      constexpr int PP = 12;  // pieces per wavefront and slab
      make_rsrc(item);
      const bool two_cols = item.valid == 0x3;
      rsrc[1] = two_cols ? rsrc[2] : (item.valid & (item.valid - 1)) ? rsrc[1] : rsrc_none;
      if (two_cols || !(item.valid & 0x5)) rsrc[2] = rsrc[3];
      // wavefronts 0, 1: the lowest unit of the mask, 2, 3: the other one, if there is one
      const int first = __builtin_ctz(item.valid), rest = item.valid & (item.valid - 1);
      const int unit = wv < 2 || !rest ? first : __builtin_ctz(rest);
      const int m0 = (unit >> 1 ? item.r[1] : item.r[0]) * kTile, n0 = (unit & 1 ? item.c[1] : item.c[0]) * kTile;
      auto barrier = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
      };
      {
        const int e0 = step_entry(0), e1 = step_entry(1), e2 = step_entry(2);
        const unsigned keep0 = keep_of(e0), keep1 = keep_of(e1);
#pragma unroll
        for (int j = 0; j < PP; ++j) gload(j, e0);
#pragma unroll
        for (int j = 0; j < PP; ++j) {
          lwrite(j, 0, keep0);
          gload(j, e1);
        }
#pragma unroll
        for (int j = 0; j < PP / 2; ++j) {
          lwrite(j, 1, keep1);
          gload(j, e2);
        }
        barrier();
      }
      // Iteration it: stage it % 2 holds slab it; beside the first substep the second half of the pieces
      // completes slab it+1 in the other stage, the barrier, beside the second the first half begins slab
      // it+2 in this one.
      if (wv >= 2 && !rest) {  // no unit: moves its pieces and keeps the barrier sequence of the others
        for (int it = 0; it < n_iter; ++it) {
          const int st = it & 1;
          const int en1 = step_entry(it + 1), en2 = step_entry(it + 2), en3 = step_entry(it + 3);
#pragma unroll
          for (int j = PP / 2; j < PP; ++j) {
            lwrite(j, st ^ 1, keep_of(en1));
            gload(j, en2);
          }
          barrier();
#pragma unroll
          for (int j = 0; j < PP / 2; ++j) {
            lwrite(j, st, keep_of(en2));
            gload(j, en3);
          }
        }
        barrier();
        barrier();
        barrier();
        return;
      }
      f32x16 acc[NT][MT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[nt][mt][i] = 0.f;
      const int a_base = (two_cols && unit == 0 ? 1 : 2) * kUnitBytes + l32 * kRowBytes;
      const int b_base = (two_cols ? 0 : wv >> 1) * kUnitBytes + l32 * kRowBytes;
      const int sub0 = 2 * (wv & 1);  // my substeps: sub0, sub0 + 1
      x8 a[2][NT], b[2][MT];
      auto lread = [&](int set, int stage, int sub, int idx) __attribute__((always_inline)) {
        const uint8_t* st = smem + stage * kStageBytes;
        const int x = rd_x ^ (sub << 5);
        if (idx == 0) {
          a[set][0] = *reinterpret_cast<const x8*>(st + a_base + x);
        } else if (idx <= MT) {
          b[set][idx - 1] = *reinterpret_cast<const x8*>(st + b_base + (idx - 1) * 32 * kRowBytes + x);
        } else {
          a[set][idx - MT] = *reinterpret_cast<const x8*>(st + a_base + (idx - MT) * 32 * kRowBytes + x);
        }
      };
      auto substep = [&](int set, int rstage, int rsub, int wstage, int j0, unsigned keep, int lentry)
                         __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NT * MT; ++i) {
          const int nt = i / MT, mt = i % MT;
          acc[nt][mt] = TT::mfma(a[set][nt], b[set][mt], acc[nt][mt]);
          if ((i & 1) == 0) {
            lread(set ^ 1, rstage, rsub, i >> 1);
          } else {
            if ((i >> 1) < PP / 2) {
              lwrite(j0 + (i >> 1), wstage, keep);
              gload(j0 + (i >> 1), lentry);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      };
#pragma unroll
      for (int idx = 0; idx < NT + MT; ++idx) lread(0, 0, sub0, idx);
      for (int it = 0; it < n_iter; ++it) {
        const int st = it & 1;
        const int en1 = step_entry(it + 1), en2 = step_entry(it + 2), en3 = step_entry(it + 3);
        substep(0, st, sub0 + 1, st ^ 1, PP / 2, keep_of(en1), en2);
        barrier();
        substep(1, st ^ 1, sub0, st, 0, keep_of(en2), en3);
      }
      barrier();
      // The two wavefronts of a unit hold sums over different k: each hands half of the rows over through
      // its quarter of the ring (32 KB, 16 bytes per lane and instruction), adds what it gets to the rows
      // it keeps, turns those as in the epilogue below and stores them.
      // (even wavefronts keep rows 0..63, odd ones 64..127: chosen value by value, a branch makes the
      // compiler copy all accumulators)
      {
        const bool odd = wv & 1;
        const int keep_row = odd ? 64 : 0;
        uint8_t* const region = smem + wv * (kSmemBytes / 4);
        const uint8_t* const other = smem + (wv ^ 1) * (kSmemBytes / 4);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
              f32x4 v;
#pragma unroll
              for (int j = 0; j < 4; ++j) v[j] = odd ? acc[nt][h][i4 * 4 + j] : acc[nt][2 + h][i4 * 4 + j];
              *reinterpret_cast<f32x4*>(region + ((h * NT + nt) * 4 + i4) * 1024 + lane * 16) = v;
              __builtin_amdgcn_sched_barrier(0);
            }
        barrier();  // every wavefront's pieces are written
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            f32x4 v[4];
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4)
              v[i4] = *reinterpret_cast<const f32x4*>(other + ((h * NT + nt) * 4 + i4) * 1024 + lane * 16);
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4)
#pragma unroll
              for (int j = 0; j < 4; ++j) acc[nt][h][i4 * 4 + j] = (odd ? acc[nt][2 + h][i4 * 4 + j] : acc[nt][h][i4 * 4 + j]) + v[i4][j];
            __builtin_amdgcn_sched_barrier(0);
          }
        barrier();  // ... and read
        const int col4 = l32;
        float bvec[4] = {0.f, 0.f, 0.f, 0.f};
        if (p.bias_kind == FO_BIAS_VECTOR) {
          const x4 bv = *reinterpret_cast<const x4*>(static_cast<const T*>(p.bias) + n0 + col4 * 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) bvec[j] = static_cast<float>(bv[j]);
        }
        const int64_t row0 = static_cast<int64_t>(item.bz) * p.m + m0;
        const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(
            static_cast<T*>(p.y) + row0 * p.n, 0, min(p.m - m0, kTile) * p.n * 2, 0x00020000);
        const int el_off = n0 + col4 * 4 + g * p.n;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint8_t* const half = region + h * (kSmemBytes / 8);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
              f32x4 v;
#pragma unroll
              for (int j = 0; j < 4; ++j) v[j] = acc[nt][h][i4 * 4 + j];
              *reinterpret_cast<f32x4*>(half + l32 * 512 + (((nt * 8 + i4 * 2 + g) ^ l32) << 4)) = v;
              __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int rk = 2 * i + g;
            const f32x4 v = *reinterpret_cast<const f32x4*>(half + rk * 512 + ((col4 ^ rk) << 4));
            x4 out;
#pragma unroll
            for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(v[j] + bvec[j]);
            typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, out), ry, el_off * 2,
                                                  (keep_row + h * 32 + 2 * i) * p.n * 2, 2);
            if ((i & 3) == 3) __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      return;
    }
  }
  int work = slot;
  bool have = work < q_len;
  Item cur{};
  // (the first slab of an item is requested before the epilogue of the item before it: its latency hides behind the stores)
  auto request_first = [&](const Item& item) {
    make_rsrc(item);
    const int e0 = step_entry(0);
#pragma unroll
    for (int j = 0; j < P; ++j) gload(j, e0);
  };
  if (have) {
    cur = decode_item(work);
    request_first(cur);
  }
  while (have) {
    const int bz = cur.bz, valid = cur.valid;
    // (no indexing by a run-time value: the item has to stay in scalar registers)
    int out_r = wr ? cur.r[1] : cur.r[0], out_c = wc ? cur.c[1] : cur.c[0];
    bool my_valid = (valid >> (wr * 2 + wc)) & 1;
    int a_tile = 2 + wc, b_tile = wr;  // LDS tiles of this wavefront's W and X operands
    if (valid & kColStrip) {
      out_r = wv == 0 ? cur.r[0] : wv == 1 ? cur.r[1] : cur.r2;
      out_c = cur.c[0];
      my_valid = wv < 3 && ((valid >> wv) & 1);
      a_tile = 2;
      b_tile = wv == 2 ? 3 : wv;
    }
    // (the next item is looked up here, while no accumulator is live)
    const int next_work = work + per_xcd;
    const bool have_next = next_work < q_len;
    Item nxt{};
    if (have_next) nxt = decode_item(next_work);
    // every wavefront is done with the ring (the previous item's epilogue turned through it)
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();

    // ---- pipeline ----
    // Two slab buffers in LDS (stage it % 2 holds slab it) and one slab in flight in the staging
    // registers.  Iteration it: substeps 0..2 of slab it run while the last three quarters of the
    // pieces of slab it+1 go from the staging registers into the other stage and the same pieces of
    // slab it+2 are requested; one barrier (every wavefront has read all of slab it and written all of
    // slab it+1); substep 3 runs while the first operands of slab it+1 are read, the first quarter of
    // slab it+2 goes into stage it % 2 and that of slab it+3 is requested.  Every substep issues the
    // same mix (sixteen MFMAs, eight operand reads, four LDS writes, four global loads), so the memory
    // path sees an even stream and a load has a whole slab period to arrive.
    {
      const int e0 = step_entry(0), e1 = step_entry(1), e2 = step_entry(2);
      {
        const unsigned keep = keep_of(e0);
#pragma unroll
        for (int j = 0; j < P; ++j) lwrite(j, 0, keep);
      }
#pragma unroll
      for (int j = 0; j < P; ++j) gload(j, e1);
      {
        const unsigned keep = keep_of(e1);
#pragma unroll
        for (int j = 0; j < PS; ++j) lwrite(j, 1, keep);
      }
#pragma unroll
      for (int j = 0; j < PS; ++j) gload(j, e2);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
    }

    auto ring_free = [&]() {
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_s_barrier();  // every wavefront is done with the ring
    };
    // ---- accumulators (the bias is added in the epilogue) ----
    // acc[nt][mt][i]: n = n0 + nt*32 + (i/4)*8 + g*4 + i%4, m = m0 + mt*32 + l32
    const int m0 = out_r * kTile;
    const int n0 = out_c * kTile;
    f32x16 acc[NT][MT];
    if (!my_valid) {
      // This wavefront's unit does not exist in this quad (unflagged, or past the matrix edge): it
      // only moves its pieces and keeps the barrier sequence of the others.
      for (int it = 0; it < n_iter; ++it) {
        const int st = it & 1;
        const int en1 = step_entry(it + 1), en2 = step_entry(it + 2), en3 = step_entry(it + 3);
        const unsigned keep1 = keep_of(en1), keep2 = keep_of(en2);
#pragma unroll
        for (int j = PS; j < P; ++j) {
          lwrite(j, st ^ 1, keep1);
          gload(j, en2);
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int j = 0; j < PS; ++j) {
          lwrite(j, st, keep2);
          gload(j, en3);
        }
      }
      ring_free();
      if (have_next) request_first(nxt);
    } else {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[nt][mt][i] = 0.f;
      {
        // LDS byte offsets of this wavefront's operand rows inside a stage
        const int a_base = a_tile * kUnitBytes + l32 * kRowBytes;  // W rows nt*32 + l32
        const int b_base = b_tile * kUnitBytes + l32 * kRowBytes;  // X rows mt*32 + l32
        x8 a[2][NT], b[2][MT];
        // operand read idx of substep sub of the slab in `stage` into register set sub & 1, in the order
        // the MFMAs need them: W rows 0, all X rows, W rows 1..3
        auto lread = [&](int stage, int sub, int idx) {
          const uint8_t* st = smem + stage * kStageBytes;
          const int x = rd_x ^ (sub << 5);
          if (idx == 0) {
            a[sub & 1][0] = *reinterpret_cast<const x8*>(st + a_base + x);
          } else if (idx <= MT) {
            b[sub & 1][idx - 1] = *reinterpret_cast<const x8*>(st + b_base + (idx - 1) * 32 * kRowBytes + x);
          } else {
            a[sub & 1][idx - MT] = *reinterpret_cast<const x8*>(st + a_base + (idx - MT) * 32 * kRowBytes + x);
          }
        };
        // one substep: the MFMAs of register set `set`; in their shadow the operand reads of substep
        // rsub of the slab in rstage, and pieces j0..j0+3: staged -> LDS stage wstage, then the same
        // pieces of the slab with entry `lentry` -> staging
        auto substep = [&](int set, int rstage, int rsub, int wstage, int j0, unsigned keep, int lentry) {
#pragma unroll
          for (int i = 0; i < NT * MT; ++i) {
            const int nt = i / MT, mt = i % MT;
            acc[nt][mt] = TT::mfma(a[set][nt], b[set][mt], acc[nt][mt]);
            if ((i & 1) == 0) lread(rstage, rsub, i >> 1);
            if ((i & 3) == 1) lwrite(j0 + (i >> 2), wstage, keep);
            if ((i & 3) == 3) gload(j0 + (i >> 2), lentry);
            __builtin_amdgcn_sched_barrier(0);
          }
        };
#pragma unroll
        for (int idx = 0; idx < NT + MT; ++idx) lread(0, 0, idx);
        int en1 = step_entry(1), en2 = step_entry(2), en3 = step_entry(3);
        for (int it = 0; it < n_iter; ++it) {
          const int st = it & 1;
          const unsigned keep1 = keep_of(en1), keep2 = keep_of(en2);
          substep(0, st, 1, st ^ 1, PS, keep1, en2);
          substep(1, st, 2, st ^ 1, 2 * PS, keep1, en2);
          substep(0, st, 3, st ^ 1, 3 * PS, keep1, en2);
          __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): my reads of slab it and my writes of slab it+1 are done
          __builtin_amdgcn_s_barrier();        // ... for every wavefront
          substep(1, st ^ 1, 0, st, 0, keep2, en3);
          en1 = en2;
          en2 = en3;
          en3 = step_entry(it + 4);
        }
      }
      ring_free();
      if (have_next) request_first(nxt);

    // ---- epilogue ----
    // In the accumulator layout a lane owns one output row and runs of four columns: written from
    // there, a store instruction is 64 scattered 8-byte pieces (measured: ~12 % of the FLUX-sized
    // launches; the bias matrix read the same way, as much again).  Each wavefront therefore turns
    // its block through its own quarter of the ring, 32 rows at a time in fp32, and adds the bias and
    // stores from a layout in which 32 consecutive lanes cover one row.
    {
      // (the lane index is made opaque: otherwise the per-lane address terms are computed once per
      // kernel, spilled, and every reload waits for the store before it)
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int col4 = ln & 31, rsub = ln >> 5, wl32 = ln & 31, wg = ln >> 5;
      uint8_t* const region0 = smem + wv * (kSmemBytes / 4);
      float bvec[4] = {0.f, 0.f, 0.f, 0.f};
      // Fused quantisation (GEMM-Q): a unit is one (token block, head) slab.  Its absmax is taken
      // over the final values (accumulator + bias, formed here in the accumulator layout without
      // being kept: the bias is added for good after the turn below); scale = absmax / 448 (1 for a
      // zero slab).
      float qscale = 1.f;
      if constexpr (kQuant) {
        {
          const bool has_vec = p.bias_kind == FO_BIAS_VECTOR;
          // all sixteen bias pieces requested before the first is used
          x4 bvs[NT * 4];
#pragma unroll
          for (int i = 0; i < NT * 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) bvs[i][j] = static_cast<T>(0.f);
          if (has_vec) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
              for (int i4 = 0; i4 < 4; ++i4)
                bvs[nt * 4 + i4] = *reinterpret_cast<const x4*>(static_cast<const T*>(p.bias) + n0 + nt * 32 +
                                                                i4 * 8 + wg * 4);
          }
          __builtin_amdgcn_sched_barrier(0);
          float amax = 0.f;
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
#pragma unroll
              for (int mt = 0; mt < MT; ++mt)
                if (m0 + mt * 32 + wl32 < p.m) {
#pragma unroll
                  for (int j = 0; j < 4; ++j) {
                    // (an opaque copy: otherwise the copies read out of the accumulator registers here
                    // are kept for the turn below, and spilled)
                    float v = acc[nt][mt][i4 * 4 + j];
                    asm volatile("" : "+v"(v));
                    amax = fmaxf(amax, fabsf(v + static_cast<float>(bvs[nt * 4 + i4][j])));
                  }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // (quarter by quarter: taken together they do not fit the registers)
          }
#pragma unroll
          for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
          qscale = amax > 0.f ? amax / 448.0f : 1.0f;
          if (lane == 0)
            p.y_scale[static_cast<int64_t>(out_c) * p.scale_row_len + bz * p.n_row_tiles + out_r] = qscale;
        }
      }
      if (p.bias_kind == FO_BIAS_VECTOR) {
        const x4 bv = *reinterpret_cast<const x4*>(static_cast<const T*>(p.bias) + n0 + col4 * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) bvec[j] = static_cast<float>(bv[j]);
      }
      // Output goes through buffer descriptors that end with the matrix: rows past M are dropped by the address
      // unit, no lane is masked and no row is tested.  A null output gets an empty descriptor.
      const int rows_out = min(p.m - m0, kTile);
      const int64_t row0 = static_cast<int64_t>(bz) * p.m + m0;
      auto out_rsrc = [&](const void* base, int elem_bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(static_cast<const uint8_t*>(base) + row0 * p.n * elem_bytes), 0,
            base ? rows_out * p.n * elem_bytes : 0, 0x00020000);
      };
      // 32 rows of the block
      auto turn_half = [&](int mt) {
        uint8_t* const region = region0 + (mt & 1) * (kSmemBytes / 8);
        // 16-byte chunk c of row r sits at chunk position c ^ r (rows are 512 bytes = 32 chunks)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int i4 = 0; i4 < 4; ++i4) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = acc[nt][mt][i4 * 4 + j];
            const int chunk = nt * 8 + i4 * 2 + wg;
            *reinterpret_cast<f32x4*>(region + wl32 * 512 + ((chunk ^ wl32) << 4)) = v;
          }
        // this lane's rows are mt*32 + rsub + 2*i, its columns n0 + col4*4 .. +3: a lane offset and a
        // scalar offset per row
        const int el_off = n0 + col4 * 4 + rsub * p.n;  // in elements, row mt*32 + rsub
        auto row_off = [&](int i, int elem_bytes) { return (mt * 32 + 2 * i) * p.n * elem_bytes; };
        const __amdgpu_buffer_rsrc_t ry = out_rsrc(p.y, 2);
        // eight rows at a time are read back (two LDS latencies per turn) and biased, then stored
        f32x4 vals[8];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if ((i & 7) == 0) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              const int rk = (i + k) * 2 + rsub;
              vals[k] = *reinterpret_cast<const f32x4*>(region + rk * 512 + ((col4 ^ rk) << 4));
            }
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) vals[i & 7][j] += bvec[j];
          const f32x4 v = vals[i & 7];
          // (stored with the streaming hint, cache policy 2: the output is not read again by this launch
          // and should not push operand tiles out of the L2; 0.5-1.5 % at both sizes)
          x4 out;
#pragma unroll
          for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(v[j]);
          typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, out), ry, el_off * 2, row_off(i, 2), 2);
          if constexpr (kQuant) {
            float f[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = fminf(fmaxf(v[j] / qscale, -448.0f), 448.0f);
            unsigned w8 = 0;
            w8 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], w8, false);
            w8 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w8, true);
            __builtin_amdgcn_raw_buffer_store_b32(w8, out_rsrc(p.y8, 1), el_off, row_off(i, 1), 0);
            typedef __attribute__((ext_vector_type(2))) float f32x2;
            const f32x2 h0 = __builtin_amdgcn_cvt_pk_f32_fp8(w8, false);
            const f32x2 h1 = __builtin_amdgcn_cvt_pk_f32_fp8(w8, true);
            unsigned l8 = 0;
            l8 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0] - h0[0], f[1] - h0[1], l8, false);
            l8 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2] - h1[0], f[3] - h1[1], l8, true);
            __builtin_amdgcn_raw_buffer_store_b32(l8, out_rsrc(p.y8_lo, 1), el_off, row_off(i, 1), 0);  // (dropped if null)
          }
        }
      };
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) turn_half(mt);
    }
    }
    cur = nxt;
    work = next_work;
    have = have_next;
  }
}

// The slabs of a token block in the order of k: the selected heads' slices (GEMM-O), or all of k.  kHalf (heads or K of 32
// mod 64): the last slab of a slice reaches 32 back, where the matrix begins, forward, and counts for one half.
struct Slab {
  uint32_t k;              // offset in bytes
  uint32_t first, second;  // masks of its halves
};
template <bool kReduce, bool kHalf>
struct SlabWalk {
  unsigned long long mask[4] = {0, 0, 0, 0};  // selected heads that are still to come
  int n_iter, iph = 1, word = 0, sub = 0, k0 = 0;

  __device__ __forceinline__ void begin(const GemmParams& p, int bz, uint32_t flag_row, int lane) {
    if constexpr (kReduce) {
      const uint8_t* info = p.sparse_info + p.sparse_info_indptr[bz];
      const bool pick = p.flag == 0;  // final pass picks bit 1, cache pass bit 0
      const int n_slices = p.k / p.head_dim;
      bool sel[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) sel[i] = 64 * i + lane < n_slices && flag_bit(info, flag_row + 64 * i + lane) == pick;
      int count = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mask[i] = __ballot(sel[i]);
        count += __popcll(mask[i]);
      }
      iph = (p.head_dim + kBK - 1) / kBK;
      n_iter = count * iph;
    } else {
      n_iter = (p.k + kBK - 1) / kBK;
    }
  }

  __device__ __forceinline__ Slab next(const GemmParams& p) {
    Slab s{0, ~0u, ~0u};
    if constexpr (kReduce) {
      if (sub == 0) {
        unsigned long long m = mask[0];
#pragma unroll
        for (int i = 1; i < 4; ++i) {
          if (m == 0 && word < i) {
            word = i;
            mask[0] = m = mask[i];
          }
        }
        k0 = (64 * word + __builtin_ctzll(m | (1ull << 63))) * p.head_dim;
        mask[0] = m & (m - 1);
      } else {
        k0 += kBK;
      }
      if (++sub == iph) sub = 0;
      s.k = static_cast<uint32_t>(k0) * 2u;
      if constexpr (kHalf) {
        if (sub == 0) {
          if (k0 >= 32) s.k -= 64u;
          (k0 >= 32 ? s.first : s.second) = 0u;
        }
      }
    } else {
      s.k = static_cast<uint32_t>(k0) * 2u;
      k0 += kBK;
      if constexpr (kHalf) {
        if (k0 > p.k) {
          s.k -= 64u;
          s.first = 0u;
        }
      }
    }
    return s;
  }
};

// Epilogue of a workgroup per unit: each wavefront turns its 64 x 64 block through 16 KB of its own (by then free) LDS in fp32,
// into a layout in which 16 consecutive lanes cover a row; bias or partial is added there, the result
// rounded once.  Output and partial go through descriptors that end with the matrix.
template <typename T, bool kReduce, bool kPartial>
__device__ __forceinline__ void unit_epilogue(const GemmParams& p, uint8_t* region, const f32x16 (&acc)[2][2], int bz, int m0,
                                              int n0, int wr, int wc, int lane) {
  using x4 = typename Types<T>::x4;
  constexpr int NT = 2, MT = 2;
  const int l32 = lane & 31, g = lane >> 5;
  const int rows_here = min(p.m - m0, kTile);
  const int col4 = lane & 15, rsub = lane >> 4;
  const int el_off = n0 + wc * 64 + col4 * 4 + (wr * 64 + rsub) * p.n;  // rows wr*64 + rsub + 4*i
  const int64_t row0 = static_cast<int64_t>(bz) * p.m + m0;
  auto out_rsrc = [&](const void* base, int elem_bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(static_cast<const uint8_t*>(base) + row0 * p.n * elem_bytes), 0,
        rows_here * p.n * elem_bytes, 0x00020000);
  };
  auto turn = [&](auto bias_tag, auto f32_tag) {
    using BiasT = decltype(bias_tag);
    using BiasVec = typename std::conditional<sizeof(BiasT) == 4, f32x4, x4>::type;
    constexpr bool kOutF32 = decltype(f32_tag)::value;
    constexpr int kBytes = sizeof(BiasT);
    // (pieces of the partial in flight together: sixteen of fp32 do not fit beside the accumulators)
    constexpr int kAhead = kBytes == 4 ? 8 : 16;
    BiasVec bm[kAhead];
    float bvec[4] = {0.f, 0.f, 0.f, 0.f};
    auto load_partial = [&](int i0) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t rb = out_rsrc(p.bias, kBytes);
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int i = i0 + k;
        if constexpr (kBytes == 4) {
          bm[k] = __builtin_bit_cast(BiasVec, __builtin_amdgcn_raw_buffer_load_b128(rb, el_off * 4, 4 * i * p.n * 4, 0));
        } else {
          bm[k] = __builtin_bit_cast(BiasVec, __builtin_amdgcn_raw_buffer_load_b64(rb, el_off * 2, 4 * i * p.n * 2, 0));
        }
      }
    };
    if constexpr (kPartial) {
      load_partial(0);
    } else if (p.bias_kind == FO_BIAS_VECTOR) {
      const x4 bv = *reinterpret_cast<const x4*>(static_cast<const T*>(p.bias) + n0 + wc * 64 + col4 * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) bvec[j] = static_cast<float>(bv[j]);
    }
    const __amdgpu_buffer_rsrc_t ry = out_rsrc(p.y, kOutF32 ? 4 : 2);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if constexpr (kPartial)
        if (mt > 0 && 8 * mt % kAhead == 0) load_partial(8 * mt);
      // 16-byte chunk c of row r sits at chunk position c ^ (r & 15) (rows are 256 bytes = 16 chunks)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          f32x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = acc[nt][mt][i4 * 4 + j];
          const int chunk = nt * 8 + i4 * 2 + g;
          *reinterpret_cast<f32x4*>(region + (mt * 32 + l32) * 256 + ((chunk ^ (l32 & 15)) << 4)) = v;
        }
      f32x4 vals[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int rk = (8 * mt + k) * 4 + rsub;
        vals[k] = *reinterpret_cast<const f32x4*>(region + rk * 256 + ((col4 ^ (rk & 15)) << 4));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int i = 8 * mt + k;
        f32x4 v = vals[k];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (kPartial) {
            v[j] += static_cast<float>(bm[i % kAhead][j]);
          } else {
            v[j] += bvec[j];
          }
        }
        if constexpr (kOutF32) {
          // (the row offset travels in the lane's: with one in a scalar register the compiler may write the first data
          // register in the very next instruction, and the last lanes then store that value)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), ry, (el_off + 4 * i * p.n) * 4, 0, 2);
        } else {
          x4 out;
#pragma unroll
          for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(v[j]);
          typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, out), ry, el_off * 2, 4 * i * p.n * 2, 2);
        }
      }
    }
  };
  using std::false_type;
  using std::true_type;
  if constexpr (!kReduce) {
    turn(T{}, false_type{});
  } else if constexpr (kPartial) {
    if (p.bias_f32) {
      if (p.y_f32) turn(0.f, true_type{}); else turn(0.f, false_type{});
    } else {
      if (p.y_f32) turn(T{}, true_type{}); else turn(T{}, false_type{});
    }
  } else {
    if (p.y_f32) turn(T{}, true_type{}); else turn(T{}, false_type{});
  }
}

// ---------------------------------------------------------------------------------------------
// One to two units per CU that are not one round of pairs (an odd number of column blocks; GEMM-O above 4096 columns): a
// workgroup per unit, two on a CU.  Quads would be one round that lasts as long however few units are in it (GEMM-Q of
// 17 000 x 384, half of the units flagged: 16.3 us, as here 10.1).  The four wavefronts share one unit (64 x 64 each: 64
// accumulators, 182 registers), two workgroups fit a CU (64 KB of LDS and GEMM-O's list), one's prologue and epilogue run
// beside the other's loop, and GEMM-O walks the heads of one token block.  The price is twice the operand bytes per flop over
// the L2 -> CU path (32 KB per 128 x 128 x 64 step, ~550 cycles of it beside 512 of matrix core), which is what bounds it.
// The loop is the quads': staging registers a slab ahead, two LDS slab buffers, one
// barrier per slab, the same mix of MFMAs, operand reads, LDS writes and loads in every substep; the
// k order is the same, and so are the results, bit for bit.
// (GEMM-O with new inputs in every call is no faster here than in the forms of longer launches: both passes of 17 000 x 384
// 21.8 us, as packed units 21.4; 1500 x 5120 103.5, as strips 98.4.)
// ---------------------------------------------------------------------------------------------
template <typename T, bool kReduce, bool kHalf, bool kPartial>
__global__ void __launch_bounds__(kThreads, 2) gemm_unit_kernel(const GemmParams p) {
  using TT = Types<T>;
  using x8 = typename TT::x8;
  using x4 = typename TT::x4;
  constexpr int NT = 2, MT = 2;  // wavefront tile: 64 columns (W rows) x 64 token rows (X rows)
  constexpr int P = 8, PS = P / 4;  // 8-row pieces per wavefront and slab (0..3 X, 4..7 W), per substep
  constexpr int kStage = 2 * kUnitBytes;  // X, W
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ int32_t s_heads[kReduce ? kMaxHeads : 1];
  __shared__ int32_t s_nsel;
  __shared__ int32_t s_step[kReduce ? kMaxSteps + 4 : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int wr = wv >> 1, wc = wv & 1;  // half of the unit's rows, of its columns

  // ---- which unit: XCD x owns the x-th eighth of the units, ordered batch, window of eight token
  // blocks, column, row: the ~64 units an XCD works on at a time share 8 + 8 operand tiles in its L2 ----
  const int units_per_batch = p.n_row_tiles * p.n_col_tiles;
  const int64_t total = static_cast<int64_t>(units_per_batch) * p.batch;
  const int xcd = blockIdx.x & (kXcds - 1), slot = blockIdx.x >> 3;
  const int u_lo = static_cast<int>(total * xcd / kXcds);
  const int u = u_lo + slot;
  if (u >= static_cast<int>(total * (xcd + 1) / kXcds)) return;
  const int bz = u / units_per_batch;
  const int rem = u - bz * units_per_batch;
  const int win = rem / (kUnitWindow * p.n_col_tiles);
  const int in_win = rem - win * kUnitWindow * p.n_col_tiles;
  const int win_rows = min(kUnitWindow, p.n_row_tiles - win * kUnitWindow);
  const int col = in_win / win_rows;
  const int row = win * kUnitWindow + in_win - col * win_rows;
  const int m0 = row * kTile, n0 = col * kTile;
  const uint32_t flag_row =
      static_cast<uint32_t>(p.num_text_tokens + m0) / static_cast<uint32_t>(p.sparse_q_size) * p.num_heads;
  if constexpr (!kReduce) {
    if (p.flag == 0) {
      const uint8_t* info = p.sparse_info + p.sparse_info_indptr[bz];
      if (!flag_bit(info, flag_row + static_cast<uint32_t>(n0) / p.head_dim)) return;
    }
  }

  // ---- k steps (entries as in gemm_kernel) ----
  int n_iter;
  if constexpr (kReduce) {
    if (wv == 0) {
      const uint8_t* info = p.sparse_info + p.sparse_info_indptr[bz];
      const bool pick = p.flag == 0;  // final pass picks bit 1, cache pass bit 0
      const int n_slices = p.k / p.head_dim;
      int count = 0;
      for (int h0 = 0; h0 < n_slices; h0 += 64) {
        const int h = h0 + lane;
        const bool sel = h < n_slices && flag_bit(info, flag_row + h) == pick;
        const unsigned long long mask = __ballot(sel);
        if (sel) s_heads[count + __popcll(mask & ((1ull << lane) - 1ull))] = h;
        count += __popcll(mask);
      }
      if (lane == 0) s_nsel = count;
    }
    __syncthreads();
    const int iph = (p.head_dim + kBK - 1) / kBK;
    n_iter = __builtin_amdgcn_readfirstlane(s_nsel) * iph;
    for (int i = tid; i < n_iter + 4 && n_iter > 0; i += kThreads) {
      const int ii = i < n_iter ? i : n_iter - 1;
      const int k0 = s_heads[ii / iph] * p.head_dim + (ii % iph) * kBK;
      int e = k0;
      if ((ii % iph) * kBK + kBK > p.head_dim) e = k0 >= 32 ? (k0 - 32) | kZeroFirst : k0 | kZeroSecond;
      s_step[i] = e;
    }
    __syncthreads();
  } else {
    n_iter = (p.k + kBK - 1) / kBK;
  }
  auto step_entry_raw = [&](int it) -> int {
    if constexpr (kReduce) {
      return s_step[it];
    } else {
      const int i = it < n_iter ? it : n_iter - 1;
      return (i + 1) * kBK <= p.k ? i * kBK : (p.k - kBK) | kZeroFirst;
    }
  };
  auto step_entry = [&](int it) -> int { return __builtin_amdgcn_readfirstlane(step_entry_raw(it)); };

  // ---- operand tiles (rows past M read as zeros through the descriptor's range check) ----
  const T* __restrict__ xg = static_cast<const T*>(p.x);
  const T* __restrict__ wg = static_cast<const T*>(p.w);
  const int rows_here = min(p.m - m0, kTile);
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(xg + (static_cast<int64_t>(bz) * p.m + m0) * p.k), 0, rows_here * p.k * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(wg + static_cast<int64_t>(n0) * p.k), 0, kTile * p.k * 2, 0x00020000);
  const int ld_chunk = lane & 7;
  int wr_off[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    wr_off[par] = (lane >> 3) * kRowBytes + ((ld_chunk ^ ((4 * par + (lane >> 4)) & 7)) << 4);
  const unsigned mask_first = ld_chunk < 4 ? 0xFFFFFFFFu : 0u;
  const int rd_x = (g ^ ((l32 >> 1) & 7)) << 4;
  int ld_off[4];
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) ld_off[jj] = (32 * wv + 8 * jj + (lane >> 3)) * p.k * 2 + ld_chunk * 16;
  u32x4 stg[P];
  auto gload = [&](int j, int entry) {
    stg[j] = __builtin_amdgcn_raw_buffer_load_b128(j < 4 ? rsrc_x : rsrc_w, ld_off[j & 3], (entry & 0xFFFF) * 2, 0);
  };
  auto keep_of = [&](int entry) -> unsigned {
    return (entry & kZeroFirst) ? ~mask_first : ((entry & kZeroSecond) ? mask_first : 0xFFFFFFFFu);
  };
  auto lwrite = [&](int j, int stage, unsigned keep) {
    uint8_t* dst = smem + stage * kStage + (j >> 2) * kUnitBytes + (32 * wv + 8 * (j & 3)) * kRowBytes + wr_off[j & 1];
    u32x4 v = stg[j];
    if constexpr (kHalf) {
      if (j < 4) v &= keep;
    }
    *reinterpret_cast<u32x4*>(dst) = v;
  };

  // acc[nt][mt][i]: column wc*64 + nt*32 + (i/4)*8 + g*4 + i%4, row wr*64 + mt*32 + l32 of the unit
  f32x16 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nt][mt][i] = 0.f;

  if (n_iter > 0) {
    const int a_base = kUnitBytes + (wc * 64 + l32) * kRowBytes;  // W rows
    const int b_base = (wr * 64 + l32) * kRowBytes;               // X rows
    // Operands are read two substeps ahead of their MFMAs (register set = substep): one ahead is 128 cycles
    // of MFMAs, less than the LDS pipe's queue of four wavefronts (256 units of K = 2048: 24.4 -> 22.5 us).
    x8 a[4][NT], b[4][MT];
    auto lread = [&](int stage, int sub, int idx) {  // W rows 0, both X row groups, W rows 1
      const uint8_t* st = smem + stage * kStage;
      const int x = rd_x ^ (sub << 5);
      if (idx == 0) {
        a[sub][0] = *reinterpret_cast<const x8*>(st + a_base + x);
      } else if (idx <= MT) {
        b[sub][idx - 1] = *reinterpret_cast<const x8*>(st + b_base + (idx - 1) * 32 * kRowBytes + x);
      } else {
        a[sub][idx - MT] = *reinterpret_cast<const x8*>(st + a_base + (idx - MT) * 32 * kRowBytes + x);
      }
    };
    auto substep = [&](int set, int rstage, int rsub, int wstage, int j0, unsigned keep, int lentry) {
#pragma unroll
      for (int i = 0; i < NT * MT; ++i) {
        const int nt = i / MT, mt = i % MT;
        acc[nt][mt] = TT::mfma(a[set][nt], b[set][mt], acc[nt][mt]);
        lread(rstage, rsub, i);
        if (i & 1) {
          lwrite(j0 + (i >> 1), wstage, keep);
          gload(j0 + (i >> 1), lentry);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int en1, en2, en3;
    {
      const int e0 = step_entry(0);
#pragma unroll
      for (int j = 0; j < P; ++j) gload(j, e0);
      en1 = step_entry(1), en2 = step_entry(2), en3 = step_entry(3);
      const unsigned keep0 = keep_of(e0), keep1 = keep_of(en1);
#pragma unroll
      for (int j = 0; j < P; ++j) {
        lwrite(j, 0, keep0);
        gload(j, en1);
      }
#pragma unroll
      for (int j = 0; j < 2 * PS; ++j) {
        lwrite(j, 1, keep1);
        gload(j, en2);
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int idx = 0; idx < NT + MT; ++idx) lread(0, sub, idx);
    // Iteration it: stage it % 2 holds slab it; substeps 0 and 1 complete slab it+1 in the other stage,
    // then (everyone has read all of slab it and written all of slab it+1) substeps 2 and 3 begin slab
    // it+2 in this one.  A piece is requested again, a slab on, once it is written.
    for (int it = 0; it < n_iter; ++it) {
      const int st = it & 1;
      const int en4_raw = step_entry_raw(it + 4);
      const unsigned keep1 = keep_of(en1), keep2 = keep_of(en2);
      substep(0, st, 2, st ^ 1, 2 * PS, keep1, en2);
      substep(1, st, 3, st ^ 1, 3 * PS, keep1, en2);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): my reads of slab it and my writes of slab it+1 are done
      __builtin_amdgcn_s_barrier();        // ... for every wavefront
      const int en4 = __builtin_amdgcn_readfirstlane(en4_raw);
      substep(2, st ^ 1, 0, st, 0, keep2, en3);
      substep(3, st ^ 1, 1, st, PS, keep2, en3);
      en1 = en2;
      en2 = en3;
      en3 = en4;
    }
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();  // every wavefront is done with the ring

  unit_epilogue<T, kReduce, kPartial>(p, smem + wv * (kUnitSmemBytes / 4), acc, bz, m0, n0, wr, wc, lane);
}

// ---------------------------------------------------------------------------------------------
// A CU for a work item: W = 1, a unit, where there is at most one per CU; W = 2, a strip of one token block x two column blocks,
// where all strips fit one round.  Nothing but the depth of an item's own pipeline hides its trips to L2 and memory then (staged
// through registers a slab ahead, as above, a unit's slab takes ~1050 cycles even on 84 of 256 CUs, 512 of them matrix core).  So
// four wavefronts per column block compute 64 x 64 each, and the rest of twelve only copy, straight to LDS, through a ring of five
// slabs of 32 KB or three of 48 KB; a copy's issue stalls (110 to 150 cycles of its wavefront) then hold up nobody's MFMAs.  With W = 2
// four copying wavefronts would be what it waits for, so each computing one issues three of a slab's 48 copies too.
// One barrier per slab, in the middle of the computation of slab t: behind it slab t + 1, which every wavefront has waited for, may
// be read, and the slab a ring further on is asked for, into the place of slab t, whose operands are all in registers by
// then (W = 1: four of the copying wavefronts are a slab behind).  Two to four (W = 2: one to two) slabs are on their way at
// any time.  The k order is that of the other forms, and so are the results, bit for bit.
// What bounds it: the copies.  Where K is a multiple of 256, the lines of a slab's rows collide somewhere on their way to the
// CU: 120 units of K = 5056 / 5120 / 5184 take 30.3 / 40.6 / 30.8 us with four copying wavefronts, 5120 33.0 with eight and 32.3
// with four of these a slab behind (eight computing wavefronts of 64 x 32: as long; other orders of k per column: as long).
// W = 1, us, two workgroups to a CU -> this, inputs of four kinds in turn, GEMM-Q flagged, dense, GEMM-O cache and final pass:
//   2 x 1100 x 1024 (144 units, 75 % flagged) 12.1 11.5 8.7 12.6 -> 10.5 10.1 8.1 10.6
//   1200 x 3072 (240, 70 %)                   26.9 28.0 17.0 25.8 -> 22.8 25.0 15.2 21.9
//   700 x 5120 (240, 70 %)                    40.7 43.0 20.1 37.6 -> 34.3 36.5 17.4 31.9
// From 257 units on it would be two rounds: 384 units of K = 3072 39.6 -> 49.7.  W = 2: see deep_strips.
// ---------------------------------------------------------------------------------------------
template <typename T, bool kReduce, bool kHalf, bool kPartial, int W>
__global__ void __launch_bounds__(kDeepThreads) gemm_deep_kernel(const GemmParams p) {
  using TT = Types<T>;
  using x8 = typename TT::x8;
  using x4 = typename TT::x4;
  constexpr int NT = 2, MT = 2;  // wavefront tile: 64 columns (W rows) x 64 token rows (X rows)
  constexpr int kCompute = 4 * W, kCopiers = kDeepThreads / 64 - kCompute, kRing = deep_ring(W);
  constexpr uint32_t kStage = (1 + W) * kUnitBytes;  // X, W of every column block
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int wr = wv / (2 * W), wc = wv % (2 * W);  // half of the rows, 64 columns

  // ---- which work item ----
  const int xcd = blockIdx.x & (kXcds - 1), slot = blockIdx.x >> 3;
  int bz, row, c0, c1 = -1;
  if constexpr (W == 1) {
    // XCD x owns the x-th eighth of the units, ordered batch, window of eight token
    // blocks, column, row: the units an XCD works on at a time share 8 + 4 operand tiles in its L2
    const int units_per_batch = p.n_row_tiles * p.n_col_tiles;
    const int64_t total = static_cast<int64_t>(units_per_batch) * p.batch;
    const int u = static_cast<int>(total * xcd / kXcds) + slot;
    if (u >= static_cast<int>(total * (xcd + 1) / kXcds)) return;
    bz = u / units_per_batch;
    const int rem = u - bz * units_per_batch;
    const int win = rem / (kUnitWindow * p.n_col_tiles);
    const int in_win = rem - win * kUnitWindow * p.n_col_tiles;
    const int win_rows = min(kUnitWindow, p.n_row_tiles - win * kUnitWindow);
    c0 = in_win / win_rows;
    row = win * kUnitWindow + in_win - c0 * win_rows;
  } else {
    // ... of the strips
    const int64_t total = static_cast<int64_t>(p.batch) * p.n_row_tiles * p.n_cp;
    const int u = static_cast<int>(total * xcd / kXcds) + slot;
    if (u >= static_cast<int>(total * (xcd + 1) / kXcds)) return;
    const int block = u / p.n_cp, cp = u - block * p.n_cp;
    bz = block / p.n_row_tiles;
    row = block - bz * p.n_row_tiles;
    c0 = 2 * cp;
    c1 = c0 + 1 < p.n_col_tiles ? c0 + 1 : -1;
  }
  bz = __builtin_amdgcn_readfirstlane(bz);
  row = __builtin_amdgcn_readfirstlane(row);
  const int m0 = row * kTile;
  const uint32_t flag_row =
      static_cast<uint32_t>(p.num_text_tokens + m0) / static_cast<uint32_t>(p.sparse_q_size) * p.num_heads;
  if constexpr (!kReduce) {
    if (p.flag == 0) {
      const uint8_t* info = p.sparse_info + p.sparse_info_indptr[bz];
      auto flagged = [&](int c) { return flag_bit(info, flag_row + static_cast<uint32_t>(c * kTile) / p.head_dim); };
      const bool f0 = flagged(c0), f1 = c1 >= 0 && flagged(max(c1, 0));
      if (!f0) c0 = -1;
      if (!f1) c1 = -1;
    }
  }
  c0 = __builtin_amdgcn_readfirstlane(c0);
  c1 = __builtin_amdgcn_readfirstlane(c1);
  if (c0 < 0 && c1 < 0) return;
  SlabWalk<kReduce, kHalf> walk;
  walk.begin(p, bz, flag_row, lane);
  const int n_iter = walk.n_iter;
  const int rows_here = min(p.m - m0, kTile);

  // ---- copies: pieces of eight rows; rows past M read as zeros through the descriptor's range check; missing column blocks
  // and slabs past the last one go through empty descriptors (zeros, no memory access) ----
  const uint32_t k2 = static_cast<uint32_t>(p.k) * 2u;
  const T* const x_base = static_cast<const T*>(p.x) + (static_cast<int64_t>(bz) * p.m + m0) * p.k;
  uint32_t voff[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    voff[par] = static_cast<uint32_t>(lane >> 3) * k2 + (((lane & 7) ^ ((4 * par + (lane >> 4)) & 7)) << 4);
  typedef __attribute__((address_space(3))) void lds_void;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)smem));
  auto copy = [&](const T* base, uint32_t bytes, uint32_t vo, uint32_t soff, uint32_t lds_addr) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, bytes, 0x00020000);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(vo), "s"(r), "s"(soff)
                 : "memory", "m0");
  };
  // of piece q of the W tiles
  auto w_base = [&](uint32_t q) __attribute__((always_inline)) -> const T* {
    return static_cast<const T*>(p.w) + static_cast<int64_t>(max(q < 16 ? c0 : c1, 0)) * kTile * p.k;
  };
  auto w_bytes = [&](uint32_t q) __attribute__((always_inline)) -> uint32_t { return (q < 16 ? c0 : c1) < 0 ? 0u : kTile * k2; };
  auto wait_copies = [&](auto n_tag) __attribute__((always_inline)) {
    constexpr int n = decltype(n_tag)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70 | (n & 15) | ((n >> 4) << 14));  // vmcnt(n)
  };
  int asked = 0;
  uint32_t at = lds0;  // where the next slab goes
  auto advance = [&]() __attribute__((always_inline)) {
    ++asked;
    at = at == lds0 + (kRing - 1) * kStage ? lds0 : at + kStage;
  };

  if (wv >= kCompute) {
    if (n_iter > 0) {
      const uint32_t cw = wv - kCompute;
      // W == 1: an eighth of the rows of either tile.  W == 2: a quarter of the pieces 8 .. 31 of the two W tiles
      constexpr int kPieces = W == 1 ? 16 / kCopiers : 24 / kCopiers, kCopies = W == 1 ? 2 * kPieces : kPieces;
      const uint32_t q0 = W == 1 ? cw * kPieces : 8 + cw * kPieces;  // (even)
      auto ask = [&]() __attribute__((always_inline)) {
        const bool live = asked < n_iter;
        const uint32_t koff = live ? walk.next(p).k : 0u;
        const uint32_t x_bytes = live ? static_cast<uint32_t>(rows_here) * k2 : 0u;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
          const uint32_t q = q0 + i;
          if constexpr (W == 1) copy(x_base, x_bytes, voff[i & 1], koff + q * 8u * k2, at + q * 8 * kRowBytes);
          copy(w_base(q), live ? w_bytes(q) : 0u, voff[i & 1], koff + (q & 15) * 8u * k2, at + kUnitBytes + q * 8 * kRowBytes);
        }
        advance();
      };
      // kLag: how many slabs this wavefront's copies are behind
      auto go = [&](auto lag_tag) __attribute__((always_inline)) {
        constexpr int kLag = decltype(lag_tag)::value;
        for (int i = 0; i < kRing - kLag; ++i) ask();
        wait_copies(std::integral_constant<int, kCopies * (kRing - 1 - kLag)>{});
        __builtin_amdgcn_s_barrier();
        for (int it = 0; it < n_iter; ++it) {
          wait_copies(std::integral_constant<int, kCopies * (kRing - 2 - kLag)>{});
          __builtin_amdgcn_s_barrier();
          ask();
        }
      };
      if (W == 2 || cw < kCopiers / 2) go(std::integral_constant<int, 0>{}); else go(std::integral_constant<int, W == 1 ? 1 : 0>{});
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): copies past the end
    __builtin_amdgcn_s_barrier();
    return;
  }

  // acc[nt][mt][i]: column wc*64 + nt*32 + (i/4)*8 + g*4 + i%4, row wr*64 + mt*32 + l32 of the item
  f32x16 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nt][mt][i] = 0.f;

  if (n_iter > 0) {
    typedef __attribute__((address_space(3))) const x8 lds_x8;
    const int rd_x = (g ^ ((l32 >> 1) & 7)) << 4;
    const uint32_t a_base = lds0 + kUnitBytes + (wc * 64 + l32) * kRowBytes;  // W rows
    const uint32_t b_base = lds0 + (wr * 64 + l32) * kRowBytes;               // X rows
    // Operands are read two substeps ahead of their MFMAs (register set = substep): one ahead is 128 cycles
    // of MFMAs, less than the LDS pipe's queue of four wavefronts.
    x8 a[4][NT], b[4][MT];
    auto lread = [&](uint32_t stage, int sub, int idx) __attribute__((always_inline)) {  // W rows 0, both X row groups, W rows 1
      const uint32_t x = stage + (rd_x ^ (sub << 5));
      if (idx == 0) {
        a[sub][0] = *reinterpret_cast<lds_x8*>(static_cast<uintptr_t>(a_base + x));
      } else if (idx <= MT) {
        b[sub][idx - 1] = *reinterpret_cast<lds_x8*>(static_cast<uintptr_t>(b_base + (idx - 1) * 32 * kRowBytes + x));
      } else {
        a[sub][idx - MT] = *reinterpret_cast<lds_x8*>(static_cast<uintptr_t>(a_base + (idx - MT) * 32 * kRowBytes + x));
      }
    };
    SlabWalk<kReduce, kHalf> mine = walk;
    Slab now{0, ~0u, ~0u};
    auto mma = [&](int sub, int i) __attribute__((always_inline)) {
      if constexpr (kHalf) {
        if (i == 0) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            b[sub][mt] = __builtin_bit_cast(x8, __builtin_bit_cast(u32x4, b[sub][mt]) & (sub < 2 ? now.first : now.second));
        }
      }
      acc[i / MT][i % MT] = TT::mfma(a[sub][i / MT], b[sub][i % MT], acc[i / MT][i % MT]);
    };
    // W == 2: two pieces of X and one of W are this wavefront's to copy
    uint32_t koff = 0, x_bytes = 0, w0_bytes = 0;
    const uint32_t voff_w = static_cast<uint32_t>(lane >> 3) * k2 + (((lane & 7) ^ ((4 * (wv & 1) + (lane >> 4)) & 7)) << 4);
    auto ask_for = [&]() __attribute__((always_inline)) {
      const bool live = asked < n_iter;
      koff = live ? walk.next(p).k : 0u;
      x_bytes = live ? static_cast<uint32_t>(rows_here) * k2 : 0u;
      w0_bytes = live ? w_bytes(0) : 0u;
    };
    auto copy_mine = [&](int i) __attribute__((always_inline)) {
      const uint32_t q = i < 2 ? 2 * wv + i : wv;
      if (i < 2) {
        copy(x_base, x_bytes, voff[i], koff + q * 8u * k2, at + q * 8 * kRowBytes);
      } else {
        copy(w_base(0), w0_bytes, voff_w, koff + q * 8u * k2, at + kUnitBytes + q * 8 * kRowBytes);
      }
    };
    if constexpr (W == 2) {
      for (int i = 0; i < kRing; ++i) {
        ask_for();
        copy_mine(0);
        copy_mine(1);
        copy_mine(2);
        advance();
      }
      wait_copies(std::integral_constant<int, 3 * (kRing - 1)>{});
    }
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int idx = 0; idx < NT + MT; ++idx) lread(0, sub, idx);
    uint32_t stage = 0;
    for (int it = 0; it < n_iter; ++it) {
      if constexpr (kHalf) now = mine.next(p);
      const uint32_t ahead = stage == (kRing - 1) * kStage ? 0u : stage + kStage;
      // substeps 0 and 1; the slab's last operand reads are three MFMAs old at the barrier
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mma(0, i);
        lread(stage, 2, i);
        if (i < 3) lread(stage, 3, i);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mma(1, i);
        if (i == 0) lread(stage, 3, 3);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (W == 2) {
        wait_copies(std::integral_constant<int, 3 * (kRing - 2)>{});
        ask_for();
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      // (behind the last slab these read what nobody uses: places of the ring that hold zeros or an older slab)
#pragma unroll
      for (int sub = 2; sub < 4; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          mma(sub, i);
          lread(ahead, sub - 2, i);
          if (W == 2 && (i == 1 || (sub == 2 && i == 3))) copy_mine(sub == 3 ? 2 : i >> 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      if constexpr (W == 2) advance();
      stage = ahead;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0)
  __builtin_amdgcn_s_barrier();  // every wavefront is done with the ring, and no copy is on its way

  const int c_mine = W == 1 || wc < 2 ? c0 : c1;
  if (c_mine < 0) return;
  unit_epilogue<T, kReduce, kPartial>(p, smem + wv * kUnitBytes, acc, bz, m0, c_mine * kTile, wr, wc & 1, lane);
}

// ---------------------------------------------------------------------------------------------
// Dense GEMM-Q whose quads leave a part of the chip idle, and narrow GEMM-O: a workgroup per unit, four of them on a CU.
// 260 quads on 256 CUs are two rounds, the second nearly empty, and 138 are one that half of the CUs sit out.  A unit per
// workgroup needs no list, and the hardware hands the next one to whichever CU is free.  What a workgroup lacks, a second
// slab buffer and staging registers, the other three on the CU make up for: a slab is copied straight to LDS (32 KB,
// one buffer), waited for, read and multiplied, and meanwhile the others are somewhere else in that cycle.
// What bounds it is LDS: 96 KB written and read per unit and slab, 750 cycles at 128 B per clock beside 512 of
// matrix core; about 920 are measured with four workgroups on every CU, against 605 per unit of a full quad.
// (Wavefronts of 64 x 128, two per workgroup, with all operands of a slab in registers need 80 KB: 710 cycles
// with four workgroups per CU, but a third slower where there are two or three; not kept.)
// us, quads -> this, dense: 2900 x 3072 (552 units) 64 -> 61; 3200 x 5120 (1000 units) 212 -> 167; 4608 x 3072 (864 units, 216 quads
// in one round) 77 -> 94.
// ---------------------------------------------------------------------------------------------
constexpr int kPackedSmemBytes = 2 * kUnitBytes;  // one slab: X, W

template <typename T, bool kReduce, bool kPartial>
__global__ void __launch_bounds__(kThreads, 4) gemm_packed_kernel(const GemmParams p) {
  using TT = Types<T>;
  using x8 = typename TT::x8;
  using x4 = typename TT::x4;
  constexpr int NT = 2, MT = 2;  // wavefront tile: 64 columns (W rows) x 64 token rows (X rows)
  constexpr int kCopies = 4;     // of X and of W each, per wavefront and slab
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  __shared__ uint16_t s_heads[kReduce ? kMaxHeads + 1 : 1];
  __shared__ int32_t s_nsel;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int wr = wv >> 1, wc = wv & 1;  // half of the unit's rows, of its columns

  // ---- which unit (order as in gemm_unit_kernel) ----
  const int units_per_batch = p.n_row_tiles * p.n_col_tiles;
  const int64_t total = static_cast<int64_t>(units_per_batch) * p.batch;
  const int xcd = blockIdx.x & (kXcds - 1), slot = blockIdx.x >> 3;
  const int u_lo = static_cast<int>(total * xcd / kXcds);
  const int u = u_lo + slot;
  if (u >= static_cast<int>(total * (xcd + 1) / kXcds)) return;
  const int bz = u / units_per_batch;
  const int rem = u - bz * units_per_batch;
  const int win = rem / (kUnitWindow * p.n_col_tiles);
  const int in_win = rem - win * kUnitWindow * p.n_col_tiles;
  const int win_rows = min(kUnitWindow, p.n_row_tiles - win * kUnitWindow);
  const int col = in_win / win_rows;
  const int row = win * kUnitWindow + in_win - col * win_rows;
  const int m0 = row * kTile, n0 = col * kTile;
  int n_iter, iph = 1;
  if constexpr (kReduce) {
    const uint32_t flag_row =
        static_cast<uint32_t>(p.num_text_tokens + m0) / static_cast<uint32_t>(p.sparse_q_size) * p.num_heads;
    if (wv == 0) {
      const uint8_t* info = p.sparse_info + p.sparse_info_indptr[bz];
      const bool pick = p.flag == 0;  // final pass picks bit 1, cache pass bit 0
      const int n_slices = p.k / p.head_dim;
      int count = 0;
      for (int h0 = 0; h0 < n_slices; h0 += 64) {
        const int h = h0 + lane;
        const bool sel = h < n_slices && flag_bit(info, flag_row + h) == pick;
        const unsigned long long mask = __ballot(sel);
        if (sel) s_heads[count + __popcll(mask & ((1ull << lane) - 1ull))] = static_cast<uint16_t>(h);
        count += __popcll(mask);
      }
      if (lane == 0) s_nsel = count;
    }
    __syncthreads();
    iph = p.head_dim / kBK;
    n_iter = __builtin_amdgcn_readfirstlane(s_nsel) * iph;
  } else {
    n_iter = p.k / kBK;
  }

  // ---- operand tiles (rows past M read as zeros through the descriptor's range check) ----
  const T* __restrict__ xg = static_cast<const T*>(p.x);
  const T* __restrict__ wg = static_cast<const T*>(p.w);
  const int rows_here = min(p.m - m0, kTile);
  const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(xg + (static_cast<int64_t>(bz) * p.m + m0) * p.k), 0, rows_here * p.k * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(wg + static_cast<int64_t>(n0) * p.k), 0, kTile * p.k * 2, 0x00020000);
  // A copy is 64 lanes x 16 bytes, global -> LDS: eight rows, lane i at row i / 8 and chunk position i % 8, where
  // logical chunk (i % 8) ^ (row / 2 % 8) belongs; row / 2 % 8 = 4 * (copy % 2) + i / 16.
  uint32_t voff[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    voff[par] = static_cast<uint32_t>((lane >> 3) * p.k * 2 + (((lane & 7) ^ ((4 * par + (lane >> 4)) & 7)) << 4));
  typedef __attribute__((address_space(3))) void lds_void;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)smem)) + wv * kCopies * 8 * kRowBytes;
  const uint32_t row_bytes8 = 8u * static_cast<uint32_t>(p.k) * 2u, wave_off = static_cast<uint32_t>(kCopies * wv) * row_bytes8;
  auto copy = [&](__amdgpu_buffer_rsrc_t rsrc, uint32_t vo, uint32_t soff, uint32_t lds_addr) __attribute__((always_inline)) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(vo), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
  };
  f32x16 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nt][mt][i] = 0.f;

  const int rd_x = (g ^ ((l32 >> 1) & 7)) << 4;
  const uint8_t* const a_base = smem + kUnitBytes + (wc * 64 + l32) * kRowBytes;  // W rows
  const uint8_t* const b_base = smem + (wr * 64 + l32) * kRowBytes;               // X rows
  // copy j of a slab: eight rows of X (the first kCopies) or of W
  auto slab_copy = [&](int j, uint32_t so) __attribute__((always_inline)) {
    const int i = j % kCopies;
    copy(j < kCopies ? rsrc_x : rsrc_w, voff[j & 1], so + i * row_bytes8, lds0 + (j < kCopies ? 0 : kUnitBytes) + i * 8 * kRowBytes);
  };
  uint32_t k0 = 0;
  int head = 0, sub = 0;
  if constexpr (kReduce) {
    if (n_iter > 0) k0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(s_heads[0])) * p.head_dim;
  }
  if (n_iter > 0) {
#pragma unroll
    for (int j = 0; j < 2 * kCopies; ++j) slab_copy(j, k0 * 2u + wave_off);
  }
  for (int it = 0; it < n_iter; ++it) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __builtin_amdgcn_s_barrier();
    x8 a[2][NT], b[2][MT];
    auto lread = [&](int ks) __attribute__((always_inline)) {
      const int x = rd_x ^ (ks << 5);
#pragma unroll
      for (int i = 0; i < NT; ++i) a[ks & 1][i] = *reinterpret_cast<const x8*>(a_base + i * 32 * kRowBytes + x);
#pragma unroll
      for (int i = 0; i < MT; ++i) b[ks & 1][i] = *reinterpret_cast<const x8*>(b_base + i * 32 * kRowBytes + x);
    };
    lread(0);
    if constexpr (kReduce) {
      if (++sub < iph) {
        k0 += kBK;
      } else {
        sub = 0;
        ++head;
        k0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(s_heads[min(head, kMaxHeads - 1)])) * p.head_dim;
      }
    } else {
      k0 += kBK;
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) {
        lread(ks + 1);
      } else {
        // every operand is in registers: the slab's place is free once that holds for every wavefront
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NT * MT; ++i) acc[i / MT][i % MT] = TT::mfma(a[ks & 1][i / MT], b[ks & 1][i % MT], acc[i / MT][i % MT]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (it + 1 < n_iter) {
#pragma unroll
      for (int j = 0; j < 2 * kCopies; ++j) slab_copy(j, k0 * 2u + wave_off);
    }
  }

  // ---- epilogue: as in gemm_unit_kernel, 32 rows at a time through a wavefront's quarter of the slab ----
  uint8_t* const region = smem + wv * (kPackedSmemBytes / 4);
  const int col4 = lane & 15, rsub = lane >> 4;
  const int el_off = n0 + wc * 64 + col4 * 4 + (wr * 64 + rsub) * p.n;  // rows wr*64 + rsub + 4*i
  const int64_t row0 = static_cast<int64_t>(bz) * p.m + m0;
  auto out_rsrc = [&](const void* base, int elem_bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(static_cast<const uint8_t*>(base) + row0 * p.n * elem_bytes), 0,
        rows_here * p.n * elem_bytes, 0x00020000);
  };
  auto turn = [&](auto bias_tag, auto f32_tag) {
    using BiasT = decltype(bias_tag);
    using BiasVec = typename std::conditional<sizeof(BiasT) == 4, f32x4, x4>::type;
    constexpr bool kOutF32 = decltype(f32_tag)::value;
    constexpr int kBytes = sizeof(BiasT);
    float bvec[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!kPartial) {
      if (p.bias_kind == FO_BIAS_VECTOR) {
        const x4 bv = *reinterpret_cast<const x4*>(static_cast<const T*>(p.bias) + n0 + wc * 64 + col4 * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) bvec[j] = static_cast<float>(bv[j]);
      }
    }
    const __amdgpu_buffer_rsrc_t ry = out_rsrc(p.y, kOutF32 ? 4 : 2);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      BiasVec bm[8];
      if constexpr (kPartial) {
        const __amdgpu_buffer_rsrc_t rb = out_rsrc(p.bias, kBytes);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int r = 4 * (8 * mt + i) * p.n;
          if constexpr (kBytes == 4) {
            bm[i] = __builtin_bit_cast(BiasVec, __builtin_amdgcn_raw_buffer_load_b128(rb, el_off * 4, r * 4, 0));
          } else {
            bm[i] = __builtin_bit_cast(BiasVec, __builtin_amdgcn_raw_buffer_load_b64(rb, el_off * 2, r * 2, 0));
          }
        }
      }
      // 16-byte chunk c of row r sits at chunk position c ^ (r & 15) (rows are 256 bytes = 16 chunks)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          f32x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = acc[nt][mt][i4 * 4 + j];
          const int chunk = nt * 8 + i4 * 2 + g;
          *reinterpret_cast<f32x4*>(region + l32 * 256 + ((chunk ^ (l32 & 15)) << 4)) = v;
        }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int rk = i * 4 + rsub;
        f32x4 v = *reinterpret_cast<const f32x4*>(region + rk * 256 + ((col4 ^ (rk & 15)) << 4));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (kPartial) {
            v[j] += static_cast<float>(bm[i][j]);
          } else {
            v[j] += bvec[j];
          }
        }
        const int r = 4 * (8 * mt + i) * p.n;
        if constexpr (kOutF32) {
          // (no scalar offset: see unit_epilogue)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), ry, (el_off + r) * 4, 0, 2);
        } else {
          x4 out;
#pragma unroll
          for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(v[j]);
          typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, out), ry, el_off * 2, r * 2, 2);
        }
      }
    }
  };
  using std::false_type;
  using std::true_type;
  if constexpr (!kReduce) {
    turn(T{}, false_type{});
  } else if constexpr (kPartial) {
    if (p.bias_f32) {
      if (p.y_f32) turn(0.f, true_type{}); else turn(0.f, false_type{});
    } else {
      if (p.y_f32) turn(T{}, true_type{}); else turn(T{}, false_type{});
    }
  } else {
    if (p.y_f32) turn(T{}, true_type{}); else turn(T{}, false_type{});
  }
}

// ---------------------------------------------------------------------------------------------
// GEMM-O: a workgroup per strip, one token block x two column blocks, two workgroups on a CU.  A strip walks its own
// block's heads (a quad walks the union of two blocks': 22.5 of 24 where each has 18, 10.5 where each has 6), and
// 864 units are 432 strips that the hardware hands out, not one round of 216 quads that lasts as long as the longest.
// A wavefront computes 64 rows x 128 columns: 128 accumulators, a slab's X operands in 32 registers, two sets of W
// operands of 32 columns; 206 registers, so two wavefronts share a SIMD and one's first touches, waits and epilogue lie
// beside the other's MFMAs.
//
// Data path.  Copies go straight to LDS, whole 128-byte lines.  A slab of W (two tiles, 32 KB) would leave no room for
// the next one beside a second workgroup, so a slab is multiplied 32 columns at a time, over all of its k, and W lives in
// a ring of six pieces of 2 x 32 rows (8 KB) of which three to five are on their way; X (16 KB) has two places: 80 KB.
// Step nt of slab t multiplies piece 4t + nt and reads piece 4t + nt + 1 (and, in its last step, X of slab t + 1, each
// register as its last MFMA is issued).  Two steps lie between barriers.  Behind the barrier in front of steps 0 and 1, when
// every wavefront has X of slab t and piece 4t in registers: pieces 4t + 5 and 4t + 6, into the places of 4t - 1 and 4t, and
// then X of slab t + 2 into that of t; in front of steps 2 and 3: pieces 4t + 7 and 4t + 8.  A piece is waited for one pair of
// steps after the pair that asked for it, X one pair later still, so eight copies may be outstanding at either barrier: X and
// two pieces behind the pieces that steps 0 and 1 read, two pieces and X behind what steps 2 and 3 do.  (X comes from memory
// when inputs are new and W from an XCD's L2: asked for half a slab later and waited for at the same barrier, X cost GEMM-Q of
// 16 384 x 3072 with a tenth flagged 56.9 us in place of 49.5, a full step of 4608 x 3072 503 in place of 494.)
// Copies past the last slab go through empty descriptors (zeros, no memory access).
//
// Order.  XCD x owns column pairs of one group and every so many-th token block (strip_cols, see launch_strips), so that
// its part of W stays in its L2; token blocks with the most selected heads come first (strip_sorted): the long ones do not end
// the launch, and those that run together walk lists of one length and stay in step, which is what keeps W in L2.  Every
// workgroup works the order out for itself (a byte or two of flags per block, one pass; ~1 us beside the other
// workgroup's loop).
//
// us, the form it replaces (quads, packed units, or both queued and one chosen on the device) -> strips, bf16: 4608 x 3072
// (24 heads), flags per head, a quarter selected 46.8 -> 31.5, three quarters 73.5 -> 66.1; a quarter of the blocks with all
// heads 59.9 -> 42.1, three quarters 72.8 -> 75.1; 33 000 x 3072 with 30 % 250 -> 192; 20 000 x 5120 with 60 % 744 -> 581;
// 76 112 x 5120 with 80 % 3105 -> 2818, with 20 % 1101 -> 871; 13 000 x 1024 with 60 % 31.4 -> 25.1.  Without the order: 36.2 (4608,
// a quarter), 670 (20 000 x 5120) and 3321 (76 112 x 5120).
//
// What bounds it: LDS and the matrix cores together (96 KB read, 48 KB written per slab of two units beside 1024 cycles of
// MFMA) and, over long launches, power: dense it takes the time of full quads to 5 % (GEMM-Q's rule in launch_q).
//
// Tiles of 16 x 16 over 32 of k: an accumulator is read and written once per 32 of k instead of once per 16, and the card
// sustains 1.98 PFLOP/s of them on random operands against 1.76 of 32 x 32 x 16 (registers only, all CUs, both at the power limit;
// with zeros both reach 2.42).  GEMM-O of 76 112 x 5120 with 80 % 2823 -> 2738 us, of 4608 x 3072, both passes, 101.2 -> 97.5.
// They are worth it where two wavefronts share a SIMD and the vector ALU has little else to issue between them: quads, one wavefront to a
// SIMD, wait for their own loads with 16 cycles of MFMA in flight instead of 32 (GEMM-Q of 76 112 x 5120 2940 -> 3230), as do
// strips of flagged units that have a CU each, which keep 32 x 32 (16 384 x 3072 with a tenth flagged, new inputs, 49.2 us, in 16 x 16
// 50.3).  The attention loop runs them in runs of sixteen, its exponentials behind them; with MFMAs and exponentials in turn, which
// want the same issue slots, they took longer there (33 k tokens x 24 heads 1709 -> 1785).
// ---------------------------------------------------------------------------------------------
constexpr int kStripPiece = 2 * 32 * kRowBytes;  // 32 rows of W of both column blocks
constexpr int kStripRing = 6;
constexpr int kStripSorted = 4096;  // token blocks that are put in order
constexpr int kStripSmemBytes = 2 * kUnitBytes + kStripRing * kStripPiece;  // 80 KB: two X tiles, the ring of W

// One strip: token block `block`, column blocks c0 and c1 (negative: none), MFMA tiles of kT x kT.
template <typename T, bool kReduce, bool kHalf, bool kPartial, int kT>
__device__ __forceinline__ void strip(const GemmParams& p, uint8_t* smem, int tid, int block, int c0, int c1) {
  using TT = Types<T>;
  using x8 = typename TT::x8;
  using x4 = typename TT::x4;
  // wavefront tile: 128 columns (W rows) x 64 token rows (X rows); a piece of W holds CT tiles of columns, a slab KS of k
  constexpr int NT = 128 / kT, MT = 64 / kT, CT = 32 / kT, KS = kT / 8, kPieces = kT * kT / 256;
  // (a descriptor has to be in scalar registers, and divisions are not)
  const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & (kT - 1), g = lane / kT;
  const int wr = wv >> 1, wc = wv & 1;  // half of the rows; column block
  block = __builtin_amdgcn_readfirstlane(block);
  c0 = __builtin_amdgcn_readfirstlane(c0);
  c1 = __builtin_amdgcn_readfirstlane(c1);
  const int bz = __builtin_amdgcn_readfirstlane(block / p.n_row_tiles), row = block - bz * p.n_row_tiles;
  const int m0 = row * kTile;
  const uint32_t flag_row = static_cast<uint32_t>(p.num_text_tokens + row * kTile) / static_cast<uint32_t>(p.sparse_q_size) * p.num_heads;

  // ---- the slabs: heads of this token block (GEMM-O), or all of k ----
  SlabWalk<kReduce, kHalf> walk;
  walk.begin(p, bz, flag_row, lane);
  const int n_iter = walk.n_iter;
  auto next_slab = [&]() __attribute__((always_inline)) -> Slab { return walk.next(p); };

  const T* __restrict__ xg = static_cast<const T*>(p.x);
  const T* __restrict__ wg = static_cast<const T*>(p.w);
  const int rows_here = min(p.m - m0, kTile);
  const uint32_t k2 = static_cast<uint32_t>(p.k) * 2u;
  const T* const x_base = xg + (static_cast<int64_t>(bz) * p.m + m0) * p.k;
  const uint32_t x_bytes = static_cast<uint32_t>(rows_here) * k2;
  // (a wavefront copies for column block wv / 2 and computes column block wv % 2)
  const int c_copy = wv >> 1 ? c1 : c0, c_mine = wc ? c1 : c0;
  const T* const w_base = wg + static_cast<int64_t>(max(c_copy, 0)) * kTile * p.k;
  const uint32_t w_bytes = c_copy < 0 ? 0u : kTile * k2;
  auto rsrc = [&](const T* base, uint32_t bytes) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, bytes, 0x00020000);
  };
  uint32_t voff[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    voff[par] = static_cast<uint32_t>(lane >> 3) * k2 + (((lane & 7) ^ ((4 * par + (lane >> 4)) & 7)) << 4);
  typedef __attribute__((address_space(3))) void lds_void;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)smem));
  const uint32_t ldsw = lds0 + 2 * kUnitBytes;  // the ring
  const uint32_t row8 = 8u * k2;
  auto copy = [&](__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t soff, uint32_t lds_addr) __attribute__((always_inline)) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(vo), "s"(r), "s"(soff)
                 : "memory", "m0");
  };
  const uint32_t x_soff = 4u * wv * row8, w_soff = 2u * (wv & 1) * row8;
  const uint32_t x_dst = lds0 + wv * 32 * kRowBytes, w_dst = ldsw + (wv >> 1) * 32 * kRowBytes + (wv & 1) * 16 * kRowBytes;
  auto copy_x = [&](__amdgpu_buffer_rsrc_t r, int i, uint32_t koff, uint32_t buf) __attribute__((always_inline)) {
    copy(r, voff[i & 1], koff + x_soff + i * row8, x_dst + buf + i * 8 * kRowBytes);
  };
  auto copy_w = [&](__amdgpu_buffer_rsrc_t r, int nt, int i, uint32_t koff, uint32_t at) __attribute__((always_inline)) {
    copy(r, voff[i & 1], koff + w_soff + (4 * nt + i) * row8, w_dst + at + i * 8 * kRowBytes);
  };

  // acc[ct][mt][i]: column ct*kT + (i/4)*8 + g*4 + i%4 of the block, row wr*64 + mt*kT + lr
  typename std::conditional<kT == 16, f32x4, f32x16>::type acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4 * kPieces; ++i) acc[nt][mt][i] = 0.f;

  if (n_iter > 0) {
    typedef __attribute__((address_space(3))) const x8 lds_x8;
    // an operand: kT rows, 512 / kT of k (ks); lane: row lr, 16-byte chunk ks*64/kT + g
    uint32_t lane_off[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      lane_off[ks] = static_cast<uint32_t>(lr * kRowBytes + (((ks * (64 / kT) + g) ^ ((lr >> 1) & 7)) << 4));
    const uint32_t x_src = lds0 + wr * 64 * kRowBytes, w_src = ldsw + wc * 32 * kRowBytes;
    x8 xr_[MT][KS], wreg[2][CT][KS];
    auto read_x = [&](int mt, int ks, uint32_t buf) __attribute__((always_inline)) {
      xr_[mt][ks] = *reinterpret_cast<lds_x8*>(static_cast<uintptr_t>(lane_off[ks] + (x_src + buf) + mt * kT * kRowBytes));
    };
    auto read_w = [&](int set, int ct, int ks, uint32_t at) __attribute__((always_inline)) {
      wreg[set][ct][ks] = *reinterpret_cast<lds_x8*>(static_cast<uintptr_t>(lane_off[ks] + (w_src + at) + ct * kT * kRowBytes));
    };
    // prologue: X of slab 0, pieces 0 to 2 | pieces 3 and 4, X of slab 1
    Slab sa = next_slab(), sb = sa;  // slabs it, it + 1
    if (n_iter > 1) sb = next_slab();
    {
      const __amdgpu_buffer_rsrc_t rx = rsrc(x_base, x_bytes), rw = rsrc(w_base, w_bytes);
      const __amdgpu_buffer_rsrc_t rx1 = rsrc(x_base, n_iter > 1 ? x_bytes : 0u), rw1 = rsrc(w_base, n_iter > 1 ? w_bytes : 0u);
#pragma unroll
      for (int i = 0; i < 4; ++i) copy_x(rx, i, sa.k, 0);
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int i = 0; i < 2; ++i) copy_w(rw, q, i, sa.k, q * kStripPiece);
#pragma unroll
      for (int i = 0; i < 4; ++i) copy_x(rx1, i, sb.k, kUnitBytes);
#pragma unroll
      for (int i = 0; i < 2; ++i) copy_w(rw, 3, i, sa.k, 3 * kStripPiece);
#pragma unroll
      for (int i = 0; i < 2; ++i) copy_w(rw1, 0, i, sb.k, 4 * kStripPiece);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70 | 8);  // vmcnt(8)
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int j = 0; j < 4; ++j) read_w(0, j % CT, j / CT, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) read_x(j % MT, j / MT, 0);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t ring = 0;  // place of the slab's first piece
    uint32_t xbuf = 0;
    auto place = [&](int j) __attribute__((always_inline)) -> uint32_t {  // of the j-th piece from the slab's first on
      uint32_t at = ring + j * kStripPiece;
      at = at >= 2 * kStripRing * kStripPiece ? at - 2 * kStripRing * kStripPiece : at;
      return at >= kStripRing * kStripPiece ? at - kStripRing * kStripPiece : at;
    };
    for (int it = 0; it < n_iter; ++it) {
      const bool live1 = it + 1 < n_iter, live2 = it + 2 < n_iter;
      Slab sc = sb;
      if (live2) sc = next_slab();
      const __amdgpu_buffer_rsrc_t rw1 = rsrc(w_base, live1 ? w_bytes : 0u);
      const __amdgpu_buffer_rsrc_t rw2 = rsrc(w_base, live2 ? w_bytes : 0u), rx2 = rsrc(x_base, live2 ? x_bytes : 0u);
      auto step = [&](auto nt_tag) __attribute__((always_inline)) {
        constexpr int nt = decltype(nt_tag)::value, set = nt & 1;
        const uint32_t rd = place(nt + 1);
        // (eighths of a step: the slots that reads and copies are dealt to)
        constexpr int kPer = CT * MT * KS / 8;
#pragma unroll
        for (int j = 0; j < 8 * kPer; ++j) {
          const int ks = j / (CT * MT), ct = j / MT % CT, mt = j % MT, slot = j / kPer;
          const bool ends = j % kPer == kPer - 1;
          if constexpr (kHalf && nt == 0) {
            if (ct == 0) {
              u32x4 v = __builtin_bit_cast(u32x4, xr_[mt][ks]);
              v &= 2 * ks < KS ? sa.first : sa.second;
              xr_[mt][ks] = __builtin_bit_cast(x8, v);
            }
          }
          if constexpr (kT == 16) {
            acc[CT * nt + ct][mt] = TT::mfma16(wreg[set][ct][ks], xr_[mt][ks], acc[CT * nt + ct][mt]);
          } else {
            acc[CT * nt + ct][mt] = TT::mfma(wreg[set][ct][ks], xr_[mt][ks], acc[CT * nt + ct][mt]);
          }
          if (slot < 4 && j % kPer == 0) read_w(set ^ 1, slot % CT, slot / CT, rd);
          if constexpr (nt == 3) {
            if constexpr (kT == 16) {
              if (ct == CT - 1) read_x(mt, ks, xbuf ^ kUnitBytes);
            } else if (mt == MT - 1) {
              read_x(0, ks, xbuf ^ kUnitBytes);
              read_x(1, ks, xbuf ^ kUnitBytes);
            }
          }
          if constexpr (nt == 0) {
            if ((slot & 1) && ends) copy_w(rw1, 1 + (slot >> 2), (slot >> 1) & 1, sb.k, place(5 + (slot >> 2)));
          } else if constexpr (nt == 1) {
            if ((slot & 1) && ends) copy_x(rx2, slot >> 1, sc.k, xbuf);
          } else {
            if ((slot == 2 || slot == 5) && ends) copy_w(nt == 2 ? rw1 : rw2, nt == 2 ? 3 : 0, slot == 5, nt == 2 ? sb.k : sc.k, place(5 + nt));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      __builtin_amdgcn_s_waitcnt(0x0f70 | 8);  // vmcnt(8)
      __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      step(std::integral_constant<int, 0>{});
      step(std::integral_constant<int, 1>{});
      __builtin_amdgcn_s_waitcnt(0x0f70 | 8);  // vmcnt(8)
      __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      step(std::integral_constant<int, 2>{});
      step(std::integral_constant<int, 3>{});
      ring = place(4);
      xbuf ^= kUnitBytes;
      sa = sb;
      sb = sc;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): copies past the end and operand reads
  __builtin_amdgcn_s_barrier();
  if (c_mine < 0) return;

  // ---- epilogue: 32 rows at a time through a wavefront's quarter of the memory ----
  uint8_t* const region = smem + wv * (kStripSmemBytes / 4);
  const int col4 = lane & 31, rsub = lane >> 5;
  const int n0 = c_mine * kTile;
  const int el_off = n0 + col4 * 4 + (wr * 64 + rsub) * p.n;  // rows wr*64 + rsub + 2*i
  const int64_t row0 = static_cast<int64_t>(bz) * p.m + m0;
  auto out_rsrc = [&](const void* base, int elem_bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(static_cast<const uint8_t*>(base) + row0 * p.n * elem_bytes), 0,
        rows_here * p.n * elem_bytes, 0x00020000);
  };
  auto turn = [&](auto bias_tag, auto f32_tag) {
    using BiasT = decltype(bias_tag);
    using BiasVec = typename std::conditional<sizeof(BiasT) == 4, f32x4, x4>::type;
    constexpr bool kOutF32 = decltype(f32_tag)::value;
    constexpr int kBytes = sizeof(BiasT);
    float bvec[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!kPartial) {
      if (p.bias_kind == FO_BIAS_VECTOR) {
        const x4 bv = *reinterpret_cast<const x4*>(static_cast<const T*>(p.bias) + n0 + col4 * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) bvec[j] = static_cast<float>(bv[j]);
      }
    }
    const __amdgpu_buffer_rsrc_t ry = out_rsrc(p.y, kOutF32 ? 4 : 2);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {  // (32 rows)
      // (rows whose partial is in flight together: sixteen of fp32 do not fit beside the accumulators)
      constexpr int kAhead = kBytes == 4 ? 8 : 16;
      BiasVec bm[kAhead];
      auto load_partial = [&](int i0) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rb = out_rsrc(p.bias, kBytes);
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          const int r = (32 * mt + 2 * (i0 + i)) * p.n;
          if constexpr (kBytes == 4) {
            bm[i] = __builtin_bit_cast(BiasVec, __builtin_amdgcn_raw_buffer_load_b128(rb, el_off * 4, r * 4, 0));
          } else {
            bm[i] = __builtin_bit_cast(BiasVec, __builtin_amdgcn_raw_buffer_load_b64(rb, el_off * 2, r * 2, 0));
          }
        }
      };
      if constexpr (kPartial) load_partial(0);
      // 16-byte chunk c of row r sits at chunk position c ^ (r & 15) (rows are 512 bytes = 32 chunks)
#pragma unroll
      for (int ct = 0; ct < NT; ++ct)
#pragma unroll
        for (int half = 0; half < 32 / kT; ++half)
#pragma unroll
          for (int i4 = 0; i4 < kPieces; ++i4) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = acc[ct][mt * (32 / kT) + half][i4 * 4 + j];
            const int r = half * kT + lr, chunk = ct * (kT / 4) + i4 * 2 + g;
            *reinterpret_cast<f32x4*>(region + r * 512 + ((chunk ^ (r & 15)) << 4)) = v;
          }
      f32x4 vals[8];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if ((i & 7) == 0) {
          if constexpr (kPartial)
            if (i > 0 && i % kAhead == 0) load_partial(i);
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const int rk = (i + k) * 2 + rsub;
            vals[k] = *reinterpret_cast<const f32x4*>(region + rk * 512 + ((col4 ^ (rk & 15)) << 4));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        f32x4 v = vals[i & 7];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (kPartial) {
            v[j] += static_cast<float>(bm[i % kAhead][j]);
          } else {
            v[j] += bvec[j];
          }
        }
        const int r = (32 * mt + 2 * i) * p.n;
        if constexpr (kOutF32) {
          // (no scalar offset: see unit_epilogue)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), ry, (el_off + r) * 4, 0, 2);
        } else {
          x4 out;
#pragma unroll
          for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(v[j]);
          typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, out), ry, el_off * 2, r * 2, 2);
        }
      }
    }
  };
  using std::false_type;
  using std::true_type;
  if constexpr (!kReduce) {
    turn(T{}, false_type{});
  } else if constexpr (kPartial) {
    if (p.bias_f32) {
      if (p.y_f32) turn(0.f, true_type{}); else turn(0.f, false_type{});
    } else {
      if (p.y_f32) turn(T{}, true_type{}); else turn(T{}, false_type{});
    }
  } else {
    if (p.y_f32) turn(T{}, true_type{}); else turn(T{}, false_type{});
  }
}

template <typename T, bool kReduce, bool kHalf, bool kPartial>
__global__ void __launch_bounds__(kThreads, 2) gemm_strip_kernel(const GemmParams p) {
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);

  if (!kReduce && p.judgement != nullptr && *p.judgement != 0) return;  // (computed as quads)
  // ---- which strip ----
  const int xcd = blockIdx.x & (kXcds - 1), slot = blockIdx.x >> 3;
  const int cols = p.strip_cols;                 // column groups of XCDs
  const int n_blocks = p.batch * p.n_row_tiles;
  auto flag_row_of = [&](int row) -> uint32_t {
    return static_cast<uint32_t>(p.num_text_tokens + row * kTile) / static_cast<uint32_t>(p.sparse_q_size) * p.num_heads;
  };
  int block, c0, c1;  // token block, column blocks (c1 < 0: only one)
  bool alone = false;  // a CU each
  if (!kReduce && p.sparse_info != nullptr) {
    // ---- GEMM-Q with flags: a token block's flagged column blocks two at a time, group of columns by group ----
    auto group_begin = [&](int g) { return g * p.n_col_tiles / cols; };
    auto flags_of = [&](int i, uint32_t* row0) -> const uint8_t* {
      const int b = i / p.n_row_tiles;
      *row0 = flag_row_of(i - b * p.n_row_tiles);
      return p.sparse_info + p.sparse_info_indptr[b];
    };
    // strips of cells first .. first + 3 (those before `end`): their flags' loads are in flight together
    constexpr int kTogether = 4;
    auto strips_of = [&](int first, int end, int (&n)[kTogether]) {
      const uint8_t* info[kTogether];
      fo::FlagRange r[kTogether];
#pragma unroll
      for (int q = 0; q < kTogether; ++q) {
        const int cell = min(first + q, end - 1), grp = cell / n_blocks;
        info[q] = flags_of(cell - grp * n_blocks, &r[q].lo);
        r[q].hi = r[q].lo + group_begin(grp + 1);
        r[q].lo += group_begin(grp);
        n[q] = 0;
      }
      if (p.head_dim == kTile) {  // (a flag per column block: four bytes of them at a time)
        for (uint32_t at0 = 0;; at0 += 4) {
          uint32_t v[kTogether][4];
          bool more = false;
#pragma unroll
          for (int q = 0; q < kTogether; ++q) {
#pragma unroll
            for (int u = 0; u < 4; ++u) v[q][u] = info[q][min(r[q].first() + at0 + u, r[q].last())];
            more |= r[q].first() + at0 + 4 <= r[q].last();
          }
#pragma unroll
          for (int q = 0; q < kTogether; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) n[q] += __popc(r[q].trim(r[q].first() + at0 + u, v[q][u]));
          if (!more) break;
        }
      } else {
#pragma unroll
        for (int q = 0; q < kTogether; ++q) {
          const uint32_t c_lo = group_begin(min(first + q, end - 1) / n_blocks), row0 = r[q].lo - c_lo;
          for (uint32_t c = c_lo; c < r[q].hi - row0; ++c) n[q] += flag_bit(info[q], row0 + c * kTile / p.head_dim);
        }
      }
#pragma unroll
      for (int q = 0; q < kTogether; ++q) n[q] = first + q < end ? (n[q] + 1) >> 1 : 0;
    };
    int32_t* const s_tot = reinterpret_cast<int32_t*>(smem);
    const int n_cells = cols * n_blocks;
    const int run = (n_cells + kThreads - 1) / kThreads;
    const int lo = min(tid * run, n_cells), hi = min(lo + run, n_cells);
    int here = 0, n[kTogether];
    for (int i = lo; i < hi; i += kTogether) {
      strips_of(i, hi, n);
#pragma unroll
      for (int q = 0; q < kTogether; ++q) here += n[q];
    }
    int upto = fo::wave_scan(here);
    if (lane == 63) s_tot[wv] = upto;
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) {
      const int t = s_tot[w];
      if (w < wv) upto += t;
      total += __builtin_amdgcn_readfirstlane(t);
    }
    alone = total <= p.num_cu;
    const int s_lo = static_cast<int>(static_cast<int64_t>(total) * xcd / kXcds);
    if (s_lo + slot >= static_cast<int>(static_cast<int64_t>(total) * (xcd + 1) / kXcds)) return;
    if (const int mine = s_lo + slot - (upto - here); mine >= 0 && mine < here) {  // (one thread)
      int skip = mine;
      for (int i = lo; i < hi; i += kTogether) {
        if (run > kTogether) strips_of(i, hi, n);  // (else they are at hand)
#pragma unroll
        for (int q = 0; q < kTogether; ++q) {
          if (skip >= 0 && skip < n[q]) {
            s_tot[8] = i + q;
            s_tot[9] = skip;
          }
          skip -= n[q];
        }
      }
    }
    __syncthreads();
    const int cell = __builtin_amdgcn_readfirstlane(s_tot[8]);
    int skip = 2 * __builtin_amdgcn_readfirstlane(s_tot[9]);
    __syncthreads();
    const int grp = cell / n_blocks, c_end = group_begin(grp + 1);
    block = cell - grp * n_blocks;
    uint32_t row0;
    const uint8_t* info = flags_of(block, &row0);
    c0 = c1 = -1;
    for (int cw = group_begin(grp); cw < c_end && c1 < 0; cw += 64) {
      const int c = min(cw + lane, c_end - 1);
      unsigned long long m = __ballot(cw + lane < c_end && flag_bit(info, row0 + static_cast<uint32_t>(c * kTile) / p.head_dim));
      if (c0 < 0 && skip >= __popcll(m)) {
        skip -= __popcll(m);
        continue;
      }
      if (c0 < 0) {
        for (; skip > 0; --skip) m &= m - 1;
        c0 = cw + __builtin_ctzll(m);
        m &= m - 1;
      }
      if (m) c1 = cw + __builtin_ctzll(m);
    }
  } else {
    const int xr = xcd / cols, xc = xcd - xr * cols;
    const int per = p.n_cp / cols;                 // column pairs of an XCD
    const int cp = xc * per + slot % per;
    block = xr + (kXcds / cols) * (slot / per);
    if (block >= n_blocks) return;
    c0 = 2 * cp;
    c1 = 2 * cp + 1 < p.n_col_tiles ? 2 * cp + 1 : -1;  // (the last pair may lack its second)
  }
  if constexpr (kReduce) {
    const int rank = block;
    if (p.strip_sorted) {
      // token blocks with the most selected heads first
      uint8_t* const s_key = smem;
      int32_t* const s_hist = reinterpret_cast<int32_t*>(smem + kStripSorted);
      const int n_slices = p.k / p.head_dim;
      if (tid < 64) s_hist[tid] = 0;
      __syncthreads();
      for (int i = tid; i < n_blocks; i += kThreads) {
        const int b = i / p.n_row_tiles;
        const uint8_t* info = p.sparse_info + p.sparse_info_indptr[b];
        const uint32_t row0 = flag_row_of(i - b * p.n_row_tiles);
        const fo::FlagRange r{row0, row0 + n_slices};
        int ones = 0;
        for (uint32_t at = r.first(); at <= r.last(); ++at) ones += __popc(r.trim(at, info[at]));
        if (p.flag) ones = n_slices - ones;
        const int key = n_slices < 64 ? ones : ones * 63 / n_slices;
        s_key[i] = static_cast<uint8_t>(key);
        atomicAdd(&s_hist[key], 1);
      }
      __syncthreads();
      const int here = s_hist[63 - lane], upto = fo::wave_scan(here);
      const unsigned long long past = __ballot(rank < upto);
      const int at = __builtin_ctzll(past), want = 63 - at;
      int skip = rank - __builtin_amdgcn_readlane(upto - here, at);
      for (int i0 = 0; i0 < n_blocks; i0 += 64) {
        unsigned long long same = __ballot(i0 + lane < n_blocks && s_key[i0 + lane] == want);
        const int n = __popcll(same);
        if (skip < n) {
          for (; skip > 0; --skip) same &= same - 1;
          block = i0 + __builtin_ctzll(same);
          break;
        }
        skip -= n;
      }
      __syncthreads();
    }
  }
  if constexpr (!kReduce) {
    if (alone) {
      strip<T, kReduce, kHalf, kPartial, 32>(p, smem, tid, block, c0, c1);
      return;
    }
  }
  strip<T, kReduce, kHalf, kPartial, 16>(p, smem, tid, block, c0, c1);
}

ListGeom make_geom(int32_t batch, int32_t m, int32_t n) {
  ListGeom gm;
  gm.batch = batch;
  gm.n_row_tiles = (m + kTile - 1) / kTile;
  gm.n_col_tiles = n / kTile;
  gm.n_win = (gm.n_row_tiles + kWindow - 1) / kWindow;
  gm.n_cp = (gm.n_col_tiles + 1) / 2;
  return gm;
}

int64_t workspace_ints(const ListGeom& gm, int64_t* max_quads_out) {
  const int64_t n_wt = static_cast<int64_t>(gm.batch) * gm.n_win, n_cells = n_wt * gm.n_cp;
  const int64_t max_quads = n_cells * kWindow;  // a cell of 16 rows x 2 columns yields at most 16 quads
  if (max_quads_out) *max_quads_out = max_quads;
  return 16 + kQuadInts * max_quads;
}

int64_t unit_count(const ListGeom& gm) { return static_cast<int64_t>(gm.batch) * gm.n_row_tiles * gm.n_col_tiles; }

// units that the rounds of quads have room for, a quad per CU and round
int64_t quad_slots(const ListGeom& gm, int num_cu) {
  const int64_t quads = static_cast<int64_t>(gm.batch) * gm.n_cp *
                        (gm.n_row_tiles / kWindow * (kWindow / 2) + (gm.n_row_tiles % kWindow + 1) / 2);
  return (quads + num_cu - 1) / num_cu * 4 * num_cu;
}

// a workgroup per unit, two on a CU
template <typename T, bool kReduce, bool kHalf, bool kAux>
int launch_units(GemmParams& p, const ListGeom& gm, hipStream_t stream) {
  static std::atomic<bool> attr_set[64] = {};
  int dev = 0;
  FO_HIP_CALL(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    FO_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_unit_kernel<T, kReduce, kHalf, kAux>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kUnitSmemBytes));
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  p.n_row_tiles = gm.n_row_tiles;
  p.n_col_tiles = gm.n_col_tiles;
  const int64_t units = unit_count(gm);
  const int64_t grid = (units + kXcds - 1) / kXcds * kXcds;
  gemm_unit_kernel<T, kReduce, kHalf, kAux><<<static_cast<unsigned>(grid), kThreads, kUnitSmemBytes, stream>>>(p);
  FO_CHECK_LAUNCH();
  return FO_OK;
}

// a workgroup per unit (W = 1) or per strip of two (W = 2), one on a CU
template <typename T, bool kReduce, bool kHalf, bool kAux, int W>
int launch_deep(GemmParams& p, const ListGeom& gm, hipStream_t stream) {
  static std::atomic<bool> attr_set[64] = {};
  int dev = 0;
  FO_HIP_CALL(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    FO_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_deep_kernel<T, kReduce, kHalf, kAux, W>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, deep_smem_bytes(W)));
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  p.n_row_tiles = gm.n_row_tiles;
  p.n_col_tiles = gm.n_col_tiles;
  p.n_cp = gm.n_cp;
  const int64_t items = static_cast<int64_t>(gm.batch) * gm.n_row_tiles * (W == 1 ? gm.n_col_tiles : gm.n_cp);
  const int64_t grid = (items + kXcds - 1) / kXcds * kXcds;
  gemm_deep_kernel<T, kReduce, kHalf, kAux, W><<<static_cast<unsigned>(grid), kDeepThreads, deep_smem_bytes(W), stream>>>(p);
  FO_CHECK_LAUNCH();
  return FO_OK;
}

// Strips of two units with a CU each, where there is more than a unit per CU and all strips fit one round.  us, units two to a
// CU -> this, inputs of four kinds in turn:
//                       GEMM-Q flagged  dense          GEMM-O cache   final
//   1500 x 3072 (288)   37.4 -> 31.9    40.7 -> 33.3   25.5 -> 22.9   31.1 -> 28.5    60 % of the heads
//   2500 x 3072 (480)   44.4 -> 40.4    48.9 -> 42.4   22.6 -> 21.5   43.7 -> 41.5    75 %
//   2 x 4000 x 1024     17.6 -> 16.1    20.7 -> 18.5   16.4 -> 15.1   19.0 -> 18.3    60 %
//   1500 x 5120 (480)   74.1 -> 58.4    82.7 -> 77.8   62.6 -> 62.9   40.2 -> 43.4    30 %
//   1000 x 5120 (320)   59.8 -> 53.4    66.1 -> 64.0   30.9 -> 29.4   55.1 -> 58.0    70 %
//   30 000 x 256 (470)   9.1 -> 9.0      9.6 -> 9.6     9.4 -> 8.6    10.0 -> 10.2    50 %
// so GEMM-Q, and GEMM-O (whose strips differ in length where units two to a CU even out) up to 4096 columns.
bool deep_strips(const ListGeom& gm, int32_t k, bool reduce, int num_cu) {
  return static_cast<int64_t>(gm.batch) * gm.n_row_tiles * gm.n_cp <= num_cu && (!reduce || k <= 4096);
}

// the same, four on a CU
template <typename T, bool kReduce, bool kAux>
int launch_packed(GemmParams& p, const ListGeom& gm, hipStream_t stream) {
  p.n_row_tiles = gm.n_row_tiles;
  p.n_col_tiles = gm.n_col_tiles;
  const int64_t units = unit_count(gm);
  const int64_t grid = (units + kXcds - 1) / kXcds * kXcds;
  gemm_packed_kernel<T, kReduce, kAux><<<static_cast<unsigned>(grid), kThreads, kPackedSmemBytes, stream>>>(p);
  FO_CHECK_LAUNCH();
  return FO_OK;
}

template <typename T, bool kReduce, bool kHalf, bool kAux>
int launch_strips(GemmParams& p, const ListGeom& gm, hipStream_t stream) {
  static std::atomic<bool> attr_set[64] = {};
  int dev = 0;
  FO_HIP_CALL(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    FO_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_strip_kernel<T, kReduce, kHalf, kAux>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kStripSmemBytes));
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  p.n_row_tiles = gm.n_row_tiles;
  p.n_col_tiles = gm.n_col_tiles;
  p.n_cp = gm.n_cp;
  // Column groups of XCDs: four, two or one that divide the column pairs and leave each at least three (20 000 x 5120, 60 % of
  // the heads: one group 734 us, two 619, four 574; 33 000 x 3072 dense 514, 499, 500).  Narrower ones are bound by memory, and
  // there a token block should be read by one XCD (60 000 x 512 dense: one group 36.8 us, two 39.4).
  // Of flagged units the strips themselves are dealt to the XCDs, an eighth each, group by group; two groups where one would
  // have more than 32 column blocks (12 000 x 5120, 20 / 50 % flagged: one group 140 / 275 us, two 130 / 267; 16 columns and
  // fewer lose up to a quarter with two).
  const bool flagged = !kReduce && p.sparse_info != nullptr;
  const int64_t rows = static_cast<int64_t>(gm.batch) * gm.n_row_tiles;
  int cols = 1;
  int64_t grid;
  if (flagged) {
    if (gm.n_col_tiles > 32) cols = 2;  // (no group is without a column)
    int64_t per = 0;  // strips of a token block, at most
    for (int g = 0; g < cols; ++g) per += ((g + 1) * gm.n_col_tiles / cols - g * gm.n_col_tiles / cols + 1) / 2;
    grid = (rows * per + kXcds - 1) / kXcds * kXcds;
  } else {
    while (cols < 4 && gm.n_cp % (2 * cols) == 0 && gm.n_cp >= 6 * cols) cols *= 2;
    const int rx = kXcds / cols;
    grid = (rows + rx - 1) / rx * (gm.n_cp / cols) * kXcds;
  }
  p.strip_cols = cols;
  p.strip_sorted = rows <= kStripSorted;
  p.num_cu = fo_num_cu();
  gemm_strip_kernel<T, kReduce, kHalf, kAux><<<static_cast<unsigned>(grid), kThreads, kStripSmemBytes, stream>>>(p);
  FO_CHECK_LAUNCH();
  return FO_OK;
}

// GEMM-O.
//   * A CU per unit or per strip (gemm_deep_kernel), then a workgroup per unit (gemm_unit_kernel), while all fit the chip at once, two
//     per CU (144 units of K = 1024: quads 28 us, units 12; strips, two workgroups to a CU, over units up to one per CU 1.3 .. 1.6, of one to two 0.91 .. 1.3, about equal from K = 1024 on).
//   * Narrow matrices, up to K = 512, are bound by memory and want the most loads in flight: packed units (strips over them,
//     three to ten units per CU: 256 columns 1.0 .. 1.3, 384 1.1 .. 1.4, 512 1.0 .. 1.1).
//   * Everything else: strips.  Over the better of quads and packed units, 2.3 to 9.7 units per CU, with 10, 50, 90 % of
//     the heads selected:
//        8 heads 0.69 .. 1.06, 0.84 .. 1.03, 0.91 .. 1.06     12  0.65 .. 0.94, 0.79 .. 0.97, 0.87 .. 1.02
//       16       0.68 .. 0.93, 0.78 .. 0.97, 0.88 .. 1.02     24  0.63 .. 0.90, 0.69 .. 1.01, 0.84 .. 1.04
//       40       0.64 .. 0.85, 0.60 .. 0.89, 0.80 .. 1.06
template <typename T, bool kHalf, bool kPartial>
int launch_o(GemmParams& p, const ListGeom& gm, hipStream_t stream) {
  const int num_cu = fo_num_cu();
  if (num_cu <= 0) return fo::fail(FO_ERR_HIP, "gemm: no device");
  if (unit_count(gm) <= num_cu) return launch_deep<T, true, kHalf, kPartial, 1>(p, gm, stream);
  if (deep_strips(gm, p.k, true, num_cu)) return launch_deep<T, true, kHalf, kPartial, 2>(p, gm, stream);
  if (unit_count(gm) <= 2 * num_cu) return launch_units<T, true, kHalf, kPartial>(p, gm, stream);
  if constexpr (!kHalf)
    if (p.k <= 512) return launch_packed<T, true, kPartial>(p, gm, stream);
  return launch_strips<T, true, kHalf, kPartial>(p, gm, stream);
}

// GEMM-Q.
//   * A CU per unit or per strip (gemm_deep_kernel), then a workgroup per unit, while all of them fit the chip at once, two
//     per CU (gemm_unit_kernel: us, quads -> units, 20 / 50 / 90 % flagged: 17 000 x 384 15.5 / 16.3 / 17.0 -> 9.6 / 10.1 / 10.8,
//     40 000 x 128, 20 / 60 %, 12.5 / 13.2 -> 6.7 / 7.0).
//   * With flags: strips from 4.5 to 32 units per CU (16 beyond 32 column blocks, whose W the strips, which drift apart,
//     read again and again; six column blocks at least, of which pairs can be made), otherwise quads, column strips and pairs
//     by the kernel's own list, whose rounds last as long however few units they hold.  Strips over those, 10 .. 95 % flagged:
//        8 heads, 4.4 to 15 units per CU  0.71 .. 1.18     16, 4.6 to 29  0.65 .. 1.05     24, 5.2 to 30  0.64 .. 1.06
//       40, 5.6 to 16                     0.66 .. 1.02         to 24      0.71 .. 1.03         to 94      1.0 .. 1.36
//     (3.4 to 4.4 units per CU 0.84 .. 1.13; 4 heads 1.1 .. 1.2).  With new inputs in every call the same, 8 to 32 heads and
//     4.9 to 29 units per CU: 0.60 .. 1.0 at most densities, but slower where the quads' last round is nearly full and strips begin
//     to share CUs (250 to 350 strips: 9000 x 3072 with 30 % 61 -> 70 us, 16 384 x 3072 with 20 % 74 -> 87, 20 000 x 1024 with 35 %
//     24 -> 28) or with most units flagged (90 %: 0.81 .. 1.12).
//   * Beyond 32 column blocks that is a wide range (8000 x 5120 from 19 to 29 % flagged, 5200 x 5120 from 30 to 47 %) and a large
//     loss, so the quads are launched first: they count, run if one round holds them, but not items of two units nor strips
//     a CU each, and leave in the scratch's first word whether they did; the strips behind them return if so.  us, strips alone ->
//     this (quads alone): 8000 x 5120, 230 strips 81 -> 84 (80), 260 121 -> 105 (103), 300 134 -> 111 (113), 345 131 -> 122 (121), 400 138 ->
//     142 (199); 5200 x 5120 80 -> 82 (81), 114 -> 100 (99), 122 -> 108 (107), 125 -> 115 (114), 133 -> 136 (204).  At 24 columns and
//     fewer the two launches cost what they give (3 us of every call; 9000 x 3072, 230 / 260 / 400 strips 50 -> 52, 71 -> 64, 82 -> 86;
//     where the quads return on a count of the flags, before any cell is walked, 1 to 4 us of every call, 8 and 16 heads gain nothing).
//   * Dense: a quad per CU and round, so it depends on how full the rounds are.  Packed units up to 21 / 32 of them (over
//     quads 0.75 .. 1.02), in a single round only up to K = 2048 (0.88 .. 1.01; 24 heads 1.05, 40 heads 1.07 .. 1.11).  Strips
//     up to K = 512 (0.87 .. 0.95 over 2.9 to 23 units per CU) and where two quads' units per CU would be empty in the last
//     of several rounds (8 heads 0.80 .. 0.87, 16 0.85 .. 0.92, 24 0.87 .. 0.95, 40 0.88 .. 0.98; fuller rounds 0.95 .. 1.09;
//     where packed units are taken they take 1.0 .. 1.2 of those' time).
//   (The fused quantiser needs a unit's absmax in one wavefront: quads only.)
template <typename T, bool kHalf, bool kQuant>
int launch_q(GemmParams& p, const ListGeom& gm, bool use_flags, void* workspace, hipStream_t stream) {
  const int num_cu = fo_num_cu();
  if (num_cu <= 0) return fo::fail(FO_ERR_HIP, "gemm: no device");
  bool strips = false;  // behind the quads, unless those run
  if constexpr (!kQuant) {
    const int64_t units = unit_count(gm);
    if (units <= num_cu) return launch_deep<T, false, kHalf, false, 1>(p, gm, stream);
    if (deep_strips(gm, p.k, false, num_cu)) return launch_deep<T, false, kHalf, false, 2>(p, gm, stream);
    if (units <= 2 * num_cu) return launch_units<T, false, kHalf, false>(p, gm, stream);
    if (use_flags && 2 * units > 9 * num_cu && units <= (gm.n_col_tiles <= 32 ? 32 : 16) * num_cu && gm.n_col_tiles >= 6) {
      if (static_cast<int64_t>(gm.batch) * gm.n_win * gm.n_cp > kInlineCells || gm.n_col_tiles <= 32)
        return launch_strips<T, false, kHalf, false>(p, gm, stream);
      strips = true;
      p.judgement = static_cast<int32_t*>(workspace);  // (its first word: no list is made here)
    }
    if (!use_flags) {
      const int64_t slots = quad_slots(gm, num_cu);
      const bool one_round = slots == 4 * num_cu;
      if constexpr (!kHalf)
        if (32 * units <= 21 * slots && (!one_round || p.k <= 2048)) return launch_packed<T, false, false>(p, gm, stream);
      if (p.k <= 512 || (!one_round && slots - units >= 2 * num_cu)) return launch_strips<T, false, kHalf, false>(p, gm, stream);
    }
  }
  // (the attribute belongs to the kernel's code object on one device: set once per device; the flags
  // are atomic because host threads may launch concurrently, and setting it twice is harmless)
  static std::atomic<bool> attr_set[64] = {};
  int dev = 0;
  FO_HIP_CALL(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    FO_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_kernel<T, kHalf, kQuant>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kSmemBytes));
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  int64_t max_quads = 0;
  workspace_ints(gm, &max_quads);
  p.n_row_tiles = gm.n_row_tiles;
  p.n_col_tiles = gm.n_col_tiles;
  p.n_cp = gm.n_cp;
  p.n_win = gm.n_win;
  p.inline_cells = 0;
  int64_t grid = (num_cu + kXcds - 1) / kXcds * kXcds;  // one persistent workgroup per CU
  const int64_t cap = (max_quads + kXcds - 1) / kXcds * kXcds;
  if (grid > cap) grid = cap;
  if (grid < kXcds) grid = kXcds;
  if (!use_flags) {
    // every unit is computed: no list, the kernel enumerates the quads itself
    p.quads = nullptr;
    p.qoff = nullptr;
    gemm_kernel<T, kHalf, kQuant><<<static_cast<unsigned>(grid), kThreads, kSmemBytes, stream>>>(p);
    FO_CHECK_LAUNCH();
    return FO_OK;
  }
  const int64_t n_cells = static_cast<int64_t>(gm.batch) * gm.n_win * gm.n_cp;
  if (n_cells <= kInlineCells) {
    // short launch: the kernel lists its quads itself (one launch less)
    p.quads = nullptr;
    p.qoff = nullptr;
    p.inline_cells = static_cast<int32_t>(n_cells);
    gemm_kernel<T, kHalf, kQuant><<<static_cast<unsigned>(grid), kThreads, kSmemBytes, stream>>>(p);
    FO_CHECK_LAUNCH();
    if constexpr (!kQuant)
      if (strips) return launch_strips<T, false, kHalf, false>(p, gm, stream);
    return FO_OK;
  }
  int32_t* qoff = static_cast<int32_t*>(workspace);
  int32_t* quads = qoff + 16;
  ListArgs la;
  la.sparse_info = p.sparse_info;
  la.sparse_info_indptr = p.sparse_info_indptr;
  la.sparse_q_size = p.sparse_q_size;
  la.num_heads = p.num_heads;
  la.head_dim = p.head_dim;
  la.num_text_tokens = p.num_text_tokens;
  gemm_quads_kernel<<<1, kListThreads, 0, stream>>>(la, gm, quads, qoff);
  FO_CHECK_LAUNCH();
  p.quads = quads;
  p.qoff = qoff;
  gemm_kernel<T, kHalf, kQuant><<<static_cast<unsigned>(grid), kThreads, kSmemBytes, stream>>>(p);
  FO_CHECK_LAUNCH();
  return FO_OK;
}

// kHalf: the k range is cut into slabs of 64 and some slab counts for one half only (GEMM-Q: K % 64 == 32;
// GEMM-O: head slices of width 32 mod 64)
template <typename T, bool kReduce>
int launch(GemmParams& p, const ListGeom& gm, bool use_flags, void* workspace, hipStream_t stream) {
  const bool half = (kReduce ? p.head_dim : p.k) % kBK != 0;
  // fused quantisation (GEMM-Q) and the cached partial (GEMM-O) get instantiations of their own, so
  // that the plain kernels do not carry their registers
  if constexpr (kReduce) {
    if (p.bias_kind == FO_BIAS_MATRIX)
      return half ? launch_o<T, true, true>(p, gm, stream) : launch_o<T, false, true>(p, gm, stream);
    return half ? launch_o<T, true, false>(p, gm, stream) : launch_o<T, false, false>(p, gm, stream);
  } else {
    if (p.y8 != nullptr)
      return half ? launch_q<T, true, true>(p, gm, use_flags, workspace, stream)
                  : launch_q<T, false, true>(p, gm, use_flags, workspace, stream);
    return half ? launch_q<T, true, false>(p, gm, use_flags, workspace, stream)
                : launch_q<T, false, false>(p, gm, use_flags, workspace, stream);
  }
}

int check_common(const void* x, const void* w, void* y, int dtype, int32_t batch, int32_t m,
                 int32_t n, int32_t k, int32_t sparse_q_size, int32_t num_qo_heads,
                 void* workspace, int64_t workspace_bytes, bool needs_list) {
  FO_REQUIRE(dtype == FO_BF16 || dtype == FO_F16, "gemm: only bf16 / fp16 operands are supported");
  FO_REQUIRE(batch > 0 && m > 0 && n > 0 && k > 0, "gemm: bad shape");
  FO_REQUIRE(n % 128 == 0 && k % 32 == 0, "only support N %% 128 == 0, K %% 32 == 0 (got N=%d K=%d)",
             n, k);
  FO_REQUIRE(k >= kBK, "gemm: K = %d is below the 64 columns one operand slab holds", k);
  FO_REQUIRE(k <= 65536, "gemm: K = %d is above 65536 (a k-step entry keeps its k offset in 16 bits)", k);
  FO_REQUIRE(sparse_q_size > 0 && num_qo_heads > 0 && n % num_qo_heads == 0,
             "gemm: bad sparse_q_size / num_qo_heads");
  FO_REQUIRE(x && w && y, "gemm: null pointer");
  FO_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) |
               reinterpret_cast<uintptr_t>(y)) & 15) == 0,
             "gemm: x, w, y must be 16-byte aligned");
  const ListGeom gm = make_geom(batch, m, n);
  FO_REQUIRE(static_cast<int64_t>(batch) * gm.n_win * gm.n_cp < (int64_t(1) << 24), "gemm: too many tiles");
  const int64_t need = 4 * workspace_ints(gm, nullptr);
  if (!needs_list) return FO_OK;  // the workspace only holds the tile list
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15))
    return fo::fail(FO_ERR_WORKSPACE, "gemm: workspace of %lld bytes (16-byte aligned) required, got %lld",
                    static_cast<long long>(need), static_cast<long long>(workspace_bytes));
  return FO_OK;
}

}  // namespace

extern "C" int64_t fo_gemm_workspace_bytes(int32_t batch, int32_t m, int32_t n) {
  if (batch <= 0 || m <= 0 || n <= 0) return 0;
  return 4 * workspace_ints(make_geom(batch, m, n), nullptr);
}

namespace {
int gemm_q_impl(const void* x, const void* w, const void* bias, void* y, uint8_t* y8, uint8_t* y8_lo,
                float* y_scale, int dtype, int32_t batch, int32_t m, int32_t n, int32_t k, int32_t sparse_q_size,
                int32_t num_qo_heads, const uint8_t* sparse_info, const int32_t* sparse_info_indptr,
                int32_t num_text_tokens, int is_full, void* workspace, int64_t workspace_bytes,
                void* stream) {
  if (int rc = check_common(x, w, y8 ? static_cast<void*>(y8) : y, dtype, batch, m, n, k, sparse_q_size,
                            num_qo_heads, workspace, workspace_bytes, !is_full))
    return rc;
  FO_REQUIRE((reinterpret_cast<uintptr_t>(y) & 15) == 0, "gemm: x, w, y must be 16-byte aligned");
  FO_REQUIRE(is_full || (sparse_info && sparse_info_indptr),
             "gemm: sparse_info and sparse_info_indptr are required unless is_full");
  FO_REQUIRE(num_text_tokens >= 0, "gemm: negative num_text_tokens");
  FO_REQUIRE(!bias || (reinterpret_cast<uintptr_t>(bias) & 7) == 0, "gemm: bias must be 8-byte aligned");
  GemmParams p{};
  p.x = x; p.w = w; p.bias = bias; p.y = y;
  p.sparse_info = is_full ? nullptr : sparse_info;
  p.sparse_info_indptr = sparse_info_indptr;
  p.batch = batch; p.m = m; p.n = n; p.k = k;
  p.sparse_q_size = sparse_q_size; p.num_heads = num_qo_heads; p.head_dim = n / num_qo_heads;
  p.num_text_tokens = num_text_tokens;
  p.flag = is_full ? 1 : 0;
  p.bias_kind = bias ? FO_BIAS_VECTOR : FO_BIAS_NONE;
  const ListGeom gm = make_geom(batch, m, n);
  if (y8) {
    FO_REQUIRE(y_scale, "gemm_q_quant: y_scale is null");
    FO_REQUIRE(p.head_dim == kTile, "gemm_q_quant: head width %d is not supported (only 128)", p.head_dim);
    FO_REQUIRE((reinterpret_cast<uintptr_t>(y8) & 3) == 0 && (reinterpret_cast<uintptr_t>(y8_lo) & 3) == 0,
               "gemm_q_quant: y8 and y8_lo must be 4-byte aligned");
    p.y8 = y8;
    p.y8_lo = y8_lo;
    p.y_scale = y_scale;
    p.scale_row_len = batch * gm.n_row_tiles;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == FO_BF16 ? launch<__bf16, false>(p, gm, !is_full, workspace, s)
                          : launch<_Float16, false>(p, gm, !is_full, workspace, s);
}
}  // namespace

extern "C" int fo_gemm_q(const void* x, const void* w, const void* bias, void* y, int dtype,
                         int32_t batch, int32_t m, int32_t n, int32_t k, int32_t sparse_q_size,
                         int32_t num_qo_heads, const uint8_t* sparse_info,
                         const int32_t* sparse_info_indptr, int32_t num_text_tokens, int is_full,
                         void* workspace, int64_t workspace_bytes, void* stream) {
  FO_REQUIRE(y, "gemm: null pointer");
  return gemm_q_impl(x, w, bias, y, nullptr, nullptr, nullptr, dtype, batch, m, n, k, sparse_q_size,
                     num_qo_heads, sparse_info, sparse_info_indptr, num_text_tokens, is_full, workspace,
                     workspace_bytes, stream);
}

extern "C" int fo_gemm_q_quant(const void* x, const void* w, const void* bias, void* y, uint8_t* y8,
                               uint8_t* y8_lo, float* y_scale, int dtype, int32_t batch, int32_t m, int32_t n,
                               int32_t k, int32_t sparse_q_size, int32_t num_qo_heads,
                               const uint8_t* sparse_info, const int32_t* sparse_info_indptr,
                               int32_t num_text_tokens, int is_full, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  FO_REQUIRE(y8, "gemm_q_quant: y8 is null");
  return gemm_q_impl(x, w, bias, y, y8, y8_lo, y_scale, dtype, batch, m, n, k, sparse_q_size, num_qo_heads,
                     sparse_info, sparse_info_indptr, num_text_tokens, is_full, workspace,
                     workspace_bytes, stream);
}

extern "C" int fo_gemm_o(const void* x, const void* w, const void* bias, void* y, int dtype,
                         int bias_kind, int bias_dtype, int y_dtype, int32_t batch, int32_t m,
                         int32_t n, int32_t k, int32_t sparse_q_size, int32_t num_qo_heads,
                         const uint8_t* sparse_info, const int32_t* sparse_info_indptr,
                         int32_t num_text_tokens, int is_for_cached, void* workspace,
                         int64_t workspace_bytes, void* stream) {
  if (int rc = check_common(x, w, y, dtype, batch, m, n, k, sparse_q_size, num_qo_heads, workspace,
                            workspace_bytes, false))
    return rc;
  FO_REQUIRE(sparse_info && sparse_info_indptr, "gemm_reduction: sparse_info is required");
  FO_REQUIRE(num_text_tokens >= 0, "gemm: negative num_text_tokens");
  const int head_dim = n / num_qo_heads;
  FO_REQUIRE(head_dim % 32 == 0 && k % head_dim == 0 && k / head_dim <= kMaxHeads && k / 32 <= kMaxSteps,
             "gemm_reduction: head slice width %d must be a multiple of 32 and divide K=%d <= 65536",
             head_dim, k);
  FO_REQUIRE(bias_kind == FO_BIAS_NONE || bias_kind == FO_BIAS_VECTOR || bias_kind == FO_BIAS_MATRIX,
             "gemm_reduction: bad bias kind");
  FO_REQUIRE(bias_kind == FO_BIAS_NONE || bias, "gemm_reduction: bias pointer is null");
  FO_REQUIRE(bias_kind != FO_BIAS_VECTOR || bias_dtype == dtype,
             "gemm_reduction: a bias vector must have the activation dtype");
  FO_REQUIRE(bias_kind != FO_BIAS_MATRIX || bias_dtype == dtype || bias_dtype == FO_F32,
             "gemm_reduction: a bias matrix must have the activation dtype or fp32");
  FO_REQUIRE(y_dtype == dtype || y_dtype == FO_F32, "gemm_reduction: bad output dtype");
  FO_REQUIRE(!bias || (reinterpret_cast<uintptr_t>(bias) & 15) == 0,
             "gemm_reduction: bias must be 16-byte aligned");
  GemmParams p{};
  p.x = x; p.w = w; p.bias = bias_kind == FO_BIAS_NONE ? nullptr : bias; p.y = y;
  p.sparse_info = sparse_info; p.sparse_info_indptr = sparse_info_indptr;
  p.batch = batch; p.m = m; p.n = n; p.k = k;
  p.sparse_q_size = sparse_q_size; p.num_heads = num_qo_heads; p.head_dim = head_dim;
  p.num_text_tokens = num_text_tokens;
  p.flag = is_for_cached ? 1 : 0;
  p.bias_kind = bias_kind;
  p.bias_f32 = bias_dtype == FO_F32;
  p.y_f32 = y_dtype == FO_F32;
  const ListGeom gm = make_geom(batch, m, n);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == FO_BF16 ? launch<__bf16, true>(p, gm, false, workspace, s)
                          : launch<_Float16, true>(p, gm, false, workspace, s);
}
