// Ragged block-sparse FlashAttention prefill for gfx950 (MI355X), driven by a decoded work list.
//
// One workgroup = 8 wavefronts (512 lanes, two per SIMD) owns one work-list row = one (request,
// 128-row q-block, head).  Wavefront w serves q rows 32*(w%4)..+31 and kv group w/4: the row's
// 64-key tiles are dealt alternately to the two kv groups, each group keeps its own running
// (max, sum, O) state and the two states are merged through LDS when the row ends.  Splitting a
// row over two kv groups halves its latency, which is what bounds the tail when there are only a
// few rows per CU, and gives every SIMD two wavefronts that are kept in opposite phases: one
// feeds the matrix cores (P.V of its previous tile, K.Q^T of its next) while the other runs its
// softmax on the vector ALUs (see the main loop).
// Only the kv blocks listed for the row are ever loaded; q-blocks that are not in the list are
// never visited, so their output bytes stay untouched.
//
// Everything is computed transposed so that no register shuffle sits between the two products:
//     S^T[kv, q] = K . Q^T        (A = K tile from LDS, B = Q kept in registers)
//     O^T[d, q] += V^T . P^T      (A = V^T via LDS transpose reads, B = P^T = exp2 of S^T, which
//                                  already has the B-operand layout)
// With v_mfma_f32_32x32x16 every lane holds one q column of S^T / O^T, so the online-softmax row
// statistics are per-lane scalars plus one exchange with lane^32.
//
// K/V tiles go global -> LDS directly (global_load_lds_dwordx4: no staging registers), two LDS
// stages per kv group; K and V of a tile are copied separately, each as soon as its half of a stage
// is free, and their completion is tracked by counting (s_waitcnt vmcnt); two barriers per
// tile.  A wavefront's 64 lanes land on 1 KB of consecutive LDS, so instead of padding the tile
// rows (256 B = 16 chunks of 16 B) are XOR-swizzled: row r keeps logical chunk c at position
// c ^ f(r), f(r) = ((r & 3) << 2) | ((r >> 2) & 3), applied on the global side of the copy.  That
// makes both the row-wise 128-bit K reads (16 consecutive rows, one chunk column) and the 4-row
// transpose reads of V (4 rows x 4 chunks) hit every bank exactly once.
//
// Work distribution: workgroups are persistent and take rows from 8 queues (one per XCD, chosen by
// blockIdx % 8) that the decoder filled head by head, so one XCD's L2 serves a few heads' K/V; the
// first row by their index, further ones from the queue's cursor; an idle XCD steals from its neighbours.
// The last workgroup to finish resets the queue cursors.  A list of at most two rows per CU is instead cut
// into one share of equal cost per workgroup, rows at the borders in parts (ranges of their kv blocks): parts
// publish unnormalised partial results to the caller's workspace and the last one to arrive combines them
// (see the end of the row loop).
//
// Between rows: while kv group 0 combines the two groups' states, one wavefront of group 1 pops the
// next item, gathers its row's metadata and copies its kv block list into LDS, so the next row
// starts with everything at hand: Q (copied into LDS like a K tile, then read as an operand) and
// the first K/V tiles are requested together.  The finished row goes through a padded LDS tile and
// leaves in 16-byte pieces, 16 consecutive lanes per 256-byte output row.  (Both were measured:
// fetched or stored from the accumulator layout, a wavefront instruction is 64 scattered pieces.)
//
// Long lists (eight rows per CU or more) run in a second form of the same kernel: a workgroup is
// 4 wavefronts that own a whole row, two such workgroups share a CU, and the main loop is software-
// pipelined in steps of 32 keys: the MFMAs of S(t+1) and P(t-1).V(t-1) and a part of the softmax of S(t) behind
// either, with the operand reads eight operands ahead and the copies two or three
// steps ahead (see the kPipe branch of the kernel).  Measured on the video-sized lists it is a quarter
// faster than the two-phase form; on short decoded lists, whose rows are taken whole, a row's doubled latency
// costs more than that.  Short lists read straight from the symbols are cut in parts as fine as it takes and run
// in it where there are enough rows (direct_pipe below); long lists of two-term fp8 q and k do
// once their k has been widened to fp16 (kWide, wide_serves).
//
// Numerics follow the reference kernel (include/flashomni/attention/prefill.cuh:759-962): base-2
// softmax p = exp2(s*c - m*c) with c = sm_scale*log2(e), P rounded to the activation type before
// P.V, row sum d over the rounded p, O = acc * rcp(d) with one round-to-nearest cast, a row with no
// kv block writes zeros and lse = -5e4 (the finite "infinity" of include/flashomni/math.cuh:32),
// lse = log2(d) + m*c.  Two liberties inside the stated tolerances: for 16-bit inputs c is
// multiplied into Q once per row (one extra rounding of q), and the reference point m is the exact
// row max of the first tile and afterwards raised only when exceeded by more than 2^8.
#include <cstdlib>
#include <type_traits>

#include "fo_common.h"
#include "fo_device.h"

namespace {

using fo::wave_max;
using fo::wave_scan;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

constexpr float kNegInf = -5e4f;  // finite "infinity" of the reference
constexpr int kThreads = 512;
constexpr int kGroupThreads = 256;
constexpr int kBlockQ = 128, kBlockKV = 128, kHeadDim = 128;
constexpr int kTileKV = 64;
constexpr int kRowBytes = 256;   // one K or V row of 128 16-bit elements, unpadded (swizzled)
constexpr int kRowBytes8 = 128;  // one fp8 K row
constexpr int kVBytes = kTileKV * kRowBytes;
constexpr int kMergeOBytes = 4 * 16 * 64 * 16;
constexpr int kOutTileOff = kMergeOBytes + 4 * 64 * 8;  // behind the merge area
constexpr int kOutRowBytes = 256 + 16;                  // one output row of 128 16-bit elements, padded
constexpr int kOutTileBytes = 128 * kOutRowBytes;
// The pipelined form's buffers of 32 keys.  K: row r keeps its 16-byte chunk c at c ^ (4 * (r % 4) + r / 4 % 4).
constexpr int kPipeKBuf = 32 * kRowBytes;
// V: every four rows (what one copy instruction fills) begin 32 bytes later modulo the banks than the four before, so that
// two 16-lane groups of a transposed read, four rows apart, meet in no bank; chunks are swizzled by the row modulo four.
constexpr int kPipeVRows4 = 4 * kRowBytes + 32, kPipeVBuf = 8 * kPipeVRows4;
// LDS geometry of one kv group: two stages of (K tile, V tile); K is 16-bit or fp8
template <bool kFp8, bool kKLo = false, int kGroups = 2>
struct Geom {
  // (fp8 K with a second term: the tile of k, then the tile of k_lo)
  static constexpr int kKBytes = kTileKV * (kFp8 ? (kKLo ? 2 : 1) * kRowBytes8 : kRowBytes);
  static constexpr int kStageBytes = kKBytes + kVBytes;
  static constexpr int kGroupBytes = 2 * kStageBytes;
  // (one kv group: eight buffers of 32 keys, see kPipeKBuf)
  static constexpr int kTilesBytes = kGroups == 1 ? 4 * (kPipeKBuf + kPipeVBuf) : kGroups * kGroupBytes;
  // the epilogue reuses the tile buffers: kv group 1's partial O (64 KB fp32) + its (max, sum)
  // pairs (2 KB), then the finished row as a padded tile for the coalesced store (one kv group:
  // no merge area, the output tile starts at 0)
  static constexpr int kOutOff = kGroups == 2 ? kOutTileOff : 0;
  static constexpr int kSmemBytes = kTilesBytes > kOutOff + kOutTileBytes ? kTilesBytes : kOutOff + kOutTileBytes;
};
constexpr int kXcds = 8;
constexpr int kMaxRowBlocks = 4096;  // kv blocks of one row held in LDS (512 Ki tokens per request)
constexpr int kMaxRowBlocksKLo = 2048;  // the same for the two-term k, whose tiles leave less LDS
constexpr int kMaxRowBlocksOneGroup = 3072;  // and for the one-group form (two workgroups share a CU's LDS)
constexpr int kMaxRowBlocksOneGroupDirect = 1024;  // where the rows' table is in LDS as well
constexpr float kLazyLog2 = 8.0f;  // the running max is raised only past a 2^8 overshoot
// merge area (reuses the tile buffers): O^T of kv group 1, then its (m, d)
static_assert(kOutTileOff + kOutTileBytes <= Geom<true>::kSmemBytes, "merge area must fit");

struct FaParams {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  float* lse;
  const void* q_lo;  // fp8: optional second e4m3 term of q (same layout and scale as q)
  const void* k_lo;  // fp8: optional second e4m3 term of k (same layout and scale as k)
  const float* q_scale;
  const float* k_scale;
  int64_t q_sn, q_sh, k_sn, k_sh, v_sn, v_sh, o_sn, o_sh;
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* q_blk_base;
  const int32_t* kv_blk_base;
  const int32_t* row_req;
  const int32_t* row_qb;
  const int32_t* row_head;
  const int32_t* kv_row_ptr;
  const int32_t* kv_idx;
  const int32_t* order;
  int32_t* sched;
  float* split_ws;  // partial results of rows whose kv list is split over workgroups (or null)
  const int32_t* shares;  // even shares: first row of every share, then the rows' cost offsets (or null)
  int32_t num_heads;
  int32_t kv_group;  // q heads per kv head (grouped-query attention); 1 = one kv head per q head
  // 0: a work-list row is (request, 128-token q block, q head).  g > 0: the reference's layout for
  // grouped-query attention with g q heads per kv head (prefill.cuh:410-413, 1283-1290): a row is
  // (request, tile, kv head), the tile being rows tile*128 .. +127 of the request's q tokens x the kv
  // head's g q heads flattened token-major (row r -> token r / g, q head kv_head * g + r % g);
  // row_head holds the kv head and kv_group is 1.
  int32_t gqa_pack;
  int32_t n_q_blocks, n_kv_blocks;  // row lengths of q_scale / k_scale
  float sm_scale_log2;
  // logits soft cap (reference: DefaultAttention, variants.cuh:43-56, :68-70): scores become
  // cap * tanh(q.k * sm_scale / cap).  cap_log2 = cap * log2(e), and sm_scale_log2 then holds
  // 2 * log2(e) * sm_scale / cap, so that exp2 of the scaled product is exp(2x) of tanh's argument.
  float cap_log2;
  // rows straight from the packed symbols (kDirect), see direct_schedule below
  const uint8_t* info;
  const uint8_t* kv_info;
  const int32_t* info_indptr;
  const int32_t* kv_info_indptr;
  const int32_t* blk_req;
  const int32_t* blk_qb;
  int32_t n_blk, batch, symbol_heads, is_full;
  int32_t zero_skipped;  // `o` is fresh: the rows of q blocks that are not computed are cleared
  // copy of the symbols for a later decode of the same rows (or null): bytes, and the two indptrs; keep_indptr
  // also where every bit counts as set (no copy): the launch marks sched[kSchedKept]
  uint8_t* keep_info;
  uint8_t* keep_kv_info;
  int32_t* keep_indptr;
  int32_t info_bytes, kv_info_bytes;
  // widened fp8 operands (see widen_k_kernel; null: none): smallest and largest k scale of every kv head, and a word
  // that the widened form sets when it has left rows to the fp8 form of the same call
  const f32x2* wide_range;
  int32_t* wide_left;
};

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
  // acc + sum of the eight elements of v (v_dot2c_f32_bf16 against ones)
  static __device__ __forceinline__ float add_elems(x8 v, float acc) {
    typedef __attribute__((ext_vector_type(2))) __bf16 x2;
    const x2 ones = {static_cast<__bf16>(1.0f), static_cast<__bf16>(1.0f)};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2_f32_bf16(x2{v[2 * i], v[2 * i + 1]}, ones, acc, false);
    return acc;
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
  static __device__ __forceinline__ float add_elems(x8 v, float acc) {
    typedef __attribute__((ext_vector_type(2))) _Float16 x2;
    const x2 ones = {static_cast<_Float16>(1.0f), static_cast<_Float16>(1.0f)};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_fdot2(x2{v[2 * i], v[2 * i + 1]}, ones, acc, false);
    return acc;
  }
};

// Whether a row runs with widened operands: the factors of its products (softmax scale c, q's scale, the k scales of its
// kv head, between range[0] and range[1]) are positive and ordinary numbers.  (False for what is not a number.)
__device__ __forceinline__ bool wide_holds(float q_scale, f32x2 range, float c) {
  const float f = c * q_scale;
  return f > 0.f && f * range[0] >= 0x1p-100f && f * range[1] <= 0x1p+90f;
}

// eight e4m3 pairs, hi + lo rounded once to fp16: both terms are multiples of 2^-9 of at most 448, so the sum is an ordinary
// fp16 number, and exact unless it takes more than 11 bits
__device__ __forceinline__ void widen8(u32x2 hi, u32x2 lo, f16x8& out) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const f32x2 h0 = __builtin_amdgcn_cvt_pk_f32_fp8(hi[j], false), h1 = __builtin_amdgcn_cvt_pk_f32_fp8(hi[j], true);
    const f32x2 l0 = __builtin_amdgcn_cvt_pk_f32_fp8(lo[j], false), l1 = __builtin_amdgcn_cvt_pk_f32_fp8(lo[j], true);
    out[4 * j + 0] = static_cast<_Float16>(h0[0] + l0[0]);
    out[4 * j + 1] = static_cast<_Float16>(h0[1] + l0[1]);
    out[4 * j + 2] = static_cast<_Float16>(h1[0] + l1[0]);
    out[4 * j + 3] = static_cast<_Float16>(h1[1] + l1[1]);
  }
}

typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void glb_void;

// chunk swizzle of a 256-byte LDS tile row r (16 chunks)
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }
// chunk swizzle of a 128-byte LDS tile row r (8 chunks; two rows span the 64 banks)
__device__ __forceinline__ int swz8(int r) { return (r >> 1) & 7; }

// 64 lanes x 16 bytes, global -> LDS: lane i fetches 16 bytes at sbase + voff and lands at LDS byte
// address lds_addr + 16*i.  sbase and lds_addr are wavefront-uniform (scalar registers), so a copy
// costs no vector-ALU work.  Issued as inline assembly on purpose: the compiler then does not
// track the copy, and does not put a vmcnt(0) in front of later LDS reads of the *other* stage that
// it cannot tell apart from the copy's destination (that wait would expose the whole copy latency
// every tile).  All waits on these copies are the explicit s_waitcnt vmcnt(0) + barrier at the
// head of a tile's MFMA block.
__device__ __forceinline__ void copy16_to_lds(const void* sbase, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_addr), "v"(voff), "s"(sbase)
               : "memory", "m0");
}

// Four 16-bit values from a 4-row x 16-column LDS patch, transposed across a 16-lane group:
// the group's lane i (0..15) supplies the address of row i/4, columns 4*(i%4)..+3, and receives
// column i of rows 0..3.
__device__ __forceinline__ s16x4 lds_read_tr16(const uint8_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
}

// max of x over lane and lane^32 (v_permlane32_swap: no LDS round trip)
__device__ __forceinline__ float max_across_halves(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const u32x2 r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  // (Each element in a scalar first: a bit cast of a vector's element reads element 0 whichever is named, and
  // then this was the maximum of the lower half.  And the instruction itself: fmaxf quiets both operands first.)
  const unsigned lo = r[0], hi = r[1];
  float m;
  asm("v_max_f32 %0, %1, %2" : "=v"(m) : "v"(lo), "v"(hi));
  return m;
}

// the same over lane and lane^16
__device__ __forceinline__ float max_across_rows(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const u32x2 r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned lo = r[0], hi = r[1];
  float m;
  asm("v_max_f32 %0, %1, %2" : "=v"(m) : "v"(lo), "v"(hi));
  return m;
}

// words of `sched` (written by the decoder): [0..8] queue bounds inside `order`, [16..23] queue
// cursors, [24] completion counter; [26] even shares in use, [27] cost share of a workgroup, [28]
// total cost, [29] number of shares, [30] number of rows, [31] the share table holds one record per
// queue entry; [64..575] arrival counters of the rows cut at share boundaries
// sched[33]: 0, or this launch's rows (1: kept symbols, 2: every row) are newer than the decoded list
constexpr int kSchedEven = 26, kSchedKept = 33, kSchedArrived = 64;
constexpr int kRecordInts = 8;  // queue entry record: row, request, q block, head, first kv slot, kv count
constexpr int kMaxShares = 512, kRowOverhead = 3, kRowOverheadPipe = 2;
constexpr int kItemBatch = 16;  // item records of a share gathered at a time
constexpr int kSplitPartFloats = 128 * 128 + 2 * 256;  // O (fp32) + (max, sum) per lane of kv group 0
// Partial results live in 2 * kMaxShares areas of the workspace: share j writes the part of a row
// that began in an earlier share to area 2j and the first part of a row that continues into the
// next share to area 2j + 1 (a share holds at most one of each).
__device__ __forceinline__ int part_area(int first_share, int part) {
  return part == 0 ? 2 * first_share + 1 : 2 * (first_share + part);
}

// Partial results cross workgroups (and XCDs, whose L2s are not coherent with each other) through
// device-scope accesses that bypass the local L2 instead of through fences, which would write back
// and invalidate a whole L2 that is busy serving K and V.
__device__ __forceinline__ void store_pair_device(float* p, float a, float b) {
  const uint64_t v = static_cast<uint64_t>(__float_as_uint(a)) | (static_cast<uint64_t>(__float_as_uint(b)) << 32);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void load_pair_device(const float* p, float& a, float& b) {
  const uint64_t v = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  a = __uint_as_float(static_cast<uint32_t>(v));
  b = __uint_as_float(static_cast<uint32_t>(v >> 32));
}

constexpr int kQueueUneven = 15;  // word of a launch's copy of the queue bounds: their lengths differ by a round or more

// Pop the next row for this workgroup from the queues, by one whole wavefront: own XCD queue first, then the
// neighbours'.  A queue's first rows belong to the workgroups of its XCD by their index and are taken without an
// atomic (see fetch_next); the cursor counts the positions behind them, which begin at `behind`.  `first` is the
// queue that this workgroup took its last row from.  When that one is empty:
//   * Queues of about one length end together, and then there is little to find: all eight cursors are looked at
//     with one load, and only a queue that still holds rows is asked.  The cursors share a cache line, whose atomics
//     are carried out one after the other (512 workgroups asking the other seven queues in turn took some 40 us at
//     the end of a launch: 512 rows of 8 kv blocks 89 -> 41 us, 1536 rows 153 -> 131; 256 workgroups: 768 rows
//     87 -> 78, 640 rows of 15 to 26 blocks 120 -> 117).
//   * Queues that differ by a round of rows or more (heads that do not divide by eight) have to be shared out in
//     any case, and the others are asked in turn, without the look: 1130 rows of 12 heads 103 -> 96 us, 1050 of 10
//     heads 78 -> 75, 790 of 6 heads 72 -> 66, 1510 rows of 12 heads on 512 workgroups 192 -> 182.
// `q` is the launch's copy of the queue bounds.  (What the workgroups of an XCD are dealt is in `behind`, in LDS, and
// not worked out from the grid's size, which is a scalar load from the launch's packet in front of every pop.)  Returns the entry's position in `order` or -1.
__device__ __forceinline__ int pop_row(const FaParams& p, int xcd, const int* q, const int* behind, int* first, int lane) {
  int a = __builtin_amdgcn_readfirstlane(*first);
  unsigned left = a < kXcds ? 1u << a : 0u;  // queues to ask, by distance from the own one
  for (bool others = false;;) {
    while (left) {
      a = __ffs(left) - 1;
      left &= left - 1;
      const int x = (xcd + a) & (kXcds - 1);
      const int beg = __builtin_amdgcn_readfirstlane(behind[x]), end = __builtin_amdgcn_readfirstlane(q[x + 1]);
      if (beg < end) {
        int pos = 0;
        if (lane == 0) pos = atomicAdd(&p.sched[16 + x], 1);
        pos = beg + __builtin_amdgcn_readfirstlane(pos);
        if (pos < end) {
          *first = a;
          return pos;
        }
      }
    }
    if (others || a >= kXcds) break;
    others = true;
    if (__builtin_amdgcn_readfirstlane(q[kQueueUneven])) {
      left = 0xffu & ~((2u << a) - 1u);
    } else {
      bool some = false;
      if (lane < kXcds) {
        const int x = (xcd + lane) & (kXcds - 1);
        const int beg = behind[x], end = q[x + 1];
        // (a cursor only grows: a queue seen empty stays empty)
        if (beg < end)
          some = beg + __hip_atomic_load(&p.sched[16 + x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < end;
      }
      left = static_cast<unsigned>(__ballot(some));
    }
  }
  *first = kXcds;
  return -1;
}

// The bits [bit, bit + n) of a byte-aligned segment as 32-bit words: word i of the range, bits outside of it
// cleared; `first` (the bit position of the range inside the first word) comes with the pointer.  Words
// are read aligned: the ends may hold bytes of the neighbouring rows, never of another allocation.
struct BitRange {
  const uint32_t* words;
  int first, n;
  // (at most 2^20 keep bits: 32-bit positions)
  __device__ __forceinline__ BitRange(const uint8_t* seg, uint32_t bit, int n_) : n(n_) {
    // (by steps from the pointer: one made from a number would be of an unknown address space, whose loads wait for LDS too)
    const uint8_t* const a = seg + (bit >> 3);
    const int skew = static_cast<int>(reinterpret_cast<uintptr_t>(a) & 3);
    words = reinterpret_cast<const uint32_t*>(a - skew);
    first = skew * 8 + static_cast<int>(bit & 7);
  }
  __device__ __forceinline__ int count() const { return (first + n + 31) >> 5; }
  __device__ __forceinline__ uint32_t trim(uint32_t v, int i) const {
    if (i == 0) v &= 0xffffffffu << first;
    const int left = first + n - 32 * i;
    if (left < 32) v &= (1u << left) - 1u;
    return v;
  }
};

// what a row's record holds besides, kDirect only (in the other kernels' records it cost the two-term fp8
// launch at 76 k tokens x 40 heads 1 %): the row's keep bits (words, position of its first bit, kv blocks
// of the request); ptr0 is then the first kept block of this part among the row's kept blocks
struct DirectMask {
  int mask;  // in words from the first whole word at or in front of the keep bits' pointer
  int mask_first, nkv;
};
struct NoMask {};
// candidates (symbol row, head): two per thread of a workgroup, four in the pipelined form, of which there are kernels for
// more (kMany: seven or eight per thread; 1000 candidates would take 61.4 us in place of 59.7 with the steps for seven, 1032 37.9 in
// place of 36.8 with those for eight; kernels for five and six of them gain nothing).  From kDirectMost + 1 on lists are long ones
// (long_list below, 256 CUs).
constexpr int kDirectMost = 2047;
// ... of which up to so many (is_full: every row is computed) may leave partial results in a workspace that other batches' launches use,
// see direct_shares_workspace
constexpr int kDirectShared = 1792, kDirectSharedFull = 1408;
constexpr int direct_max_cand(int many) { return many == 0 ? 1024 : 256 * many < kDirectMost ? 256 * many : kDirectMost; }
constexpr int kDirectShareRows = 1024;  // rows of a share that the table of them holds (see direct_table_holds)
constexpr int kDirectMaxParts = 8;    // parts of a row, one workgroup each
constexpr int kDirectMapBytes = (1 << 16) - 16;  // keep bits that are staged in the tile buffers (both forms have as much)
constexpr int kOlderGain = 4;  // see cut_at
constexpr int kPartExtra = 2, kEvenExtra = 5;  // what cutting rows costs a workgroup, in kv blocks (see direct_schedule)
constexpr int kDirectMinPart = 4;     // kv blocks that a part is worth: prologue, epilogue and exchange cost about as many

// T: element type of V, P and O (and of Q, K unless kFp8).  kFp8: Q and K are e4m3fn bytes with one
// dequantisation scale per (head, 128-token block); S^T then comes from
// v_mfma_scale_f32_32x32x64_f8f6f4 (64 d per instruction, unit block scale) and the two per-block
// scales are folded into the softmax scale of the tile.  kQLo: q comes as two e4m3 terms, q + q_lo
// (the second one the rounding residual of the first), and S^T = K.(q + q_lo)^T takes two MFMAs
// per slab: e4m3 keeps 3 mantissa bits, and with both operands rounded to it the logits are too
// noisy for the accuracy this path promises; with the two-term q only k's rounding is left.  The
// fp8 matrix cores run at twice the 16-bit rate, so the two terms cost what a 16-bit S^T costs.
// kKLo: k comes as two e4m3 terms as well, k + k_lo; S^T = k.q^T + k.q_lo^T + k_lo.q^T (the product
// of the two residuals, 2^-8 of the logit, is left out): both operands then carry ~7 significant
// bits and the logits are as accurate as 16-bit ones.  This is the accuracy form, not a fast one.  Long lists of
// such operands run with both widened to fp16 where there is room for it (kWide, see widen_k_kernel): one product.
//
// kGroups: kv groups of a workgroup.  2: the form described at the top of this file (8 wavefronts).
// 1: a workgroup is 4 wavefronts (q sub-tiles 0..3) that walk all tiles of the row, two such
// workgroups share a CU (one wavefront of each per SIMD) and run independent rows: nothing ties
// their phases together, there is no merge, and one's row prologue / epilogue overlaps the other's
// main loop.  A row takes twice as long, so this is the form for long lists (many rows per CU).
template <typename T, bool kFp8, bool kQLo, bool kKLo, int kGroups, bool kPipe = false, bool kGqaPack = false,
          bool kCap = false, bool kDirect = false, bool kWide = false, int kMany = 0>
__global__ void __launch_bounds__(kGroups * kGroupThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
sparse_fa_kernel(const FaParams p) {
  static_assert(!kWide || (kPipe && !kGqaPack && !kDirect), "widened operands are a variant of the pipelined loop");
  static_assert(kPipe == (kGroups == 1), "one kv group runs the software-pipelined loop, two the two-phase loop");
  static_assert(!kPipe || !kFp8, "the software-pipelined loop is built for 16-bit operands");
  static_assert(kFp8 || !kQLo, "the two-term q is an fp8 form");
  static_assert(kQLo || !kKLo, "the two-term k is built on the two-term q");
  static_assert(!kCap || (!kFp8 && !kPipe), "the logits soft cap is built into the two-phase loop for 16-bit operands");
  constexpr int kWaves = 4 * kGroups;
  constexpr int kShareRowCost = kPipe ? kRowOverheadPipe : kRowOverhead;  // kDirect: what a row costs beside its kv blocks
  constexpr int kFetchWave = kGroups == 2 ? 4 : 0;  // the wavefront that fetches the next item
  using TT = Types<T>;
  using TS = Types<typename std::conditional<kWide, _Float16, T>::type>;  // Q and K
  using q8 = typename TS::x8;
  using x8 = typename TT::x8;
  using x4 = typename TT::x4;
  using G = Geom<kFp8, kKLo, kGroups>;
  using TQK = typename std::conditional<kFp8, uint8_t, T>::type;
  constexpr int kStageBytes = G::kStageBytes, kKBytes = G::kKBytes, kGroupBytes = G::kGroupBytes;
  // (256-byte aligned: lane offsets with XOR-swizzled low bits can then carry the array's base)
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  // this item / the next one, with everything the row's prologue needs: fetched by the popping lane
  // while the rest of the workgroup finishes the current row
  struct RowInfo : std::conditional<kDirect, DirectMask, NoMask>::type {
    int row, part, parts, slot, req, qb, head, q_begin, q_rows, kv_begin, kv_len, ptr0, nb;
    float q_scale;  // fp8: dequantisation scale of the row's q block
    int k_scale0;   // fp8: position of the request's first kv block in k_scale (the kv head's row); kWide: in k16
  };
  // (fetched with the rest of the record: read in the row's prologue, they would wait behind every
  // tile copy in flight)
  auto fill_scales = [&](RowInfo& it) {
    it.q_scale = 1.f;
    it.k_scale0 = 0;
    if constexpr (kFp8 || kWide)
      it.q_scale = p.q_scale[static_cast<int64_t>(it.head) * p.n_q_blocks + p.q_blk_base[it.req] + it.qb];
    if constexpr (kFp8 || kWide) it.k_scale0 = (it.head / p.kv_group) * p.n_kv_blocks + p.kv_blk_base[it.req];
  };
  // q_begin: first token of the item's q rows; q_rows: how many of its 128 rows exist
  auto set_q_range = [&](RowInfo& it, const int32_t* ends) {
    const int q0 = ends[0], q1 = ends[1];
    if (kGqaPack) {  // (rows are (token, q head) pairs counted from the request's first token)
      it.q_begin = q0;
      it.q_rows = min(kBlockQ, (q1 - q0) * p.gqa_pack - it.qb * kBlockQ);
    } else {
      it.q_begin = q0 + it.qb * kBlockQ;
      it.q_rows = min(kBlockQ, q1 - it.q_begin);
    }
  };
  __shared__ RowInfo s_next_row[2];
  __shared__ int s_arrived;
  __shared__ int s_behind[kXcds];  // the position of every queue behind the rows that are dealt
  __shared__ int s_queue[16];  // queue bounds and even-share words of `sched`, read once
  __shared__ int s_share[1];   // even shares: items of this workgroup's share handed out so far
  __shared__ int s_guess;      // queues: one past the position this workgroup popped last
  __shared__ RowInfo s_items[kItemBatch];  // even shares: records of the share's next items
  constexpr int kRowBlocks = kGroups == 1 ? (kDirect ? kMaxRowBlocksOneGroupDirect : kMaxRowBlocksOneGroup)
                             : kKLo       ? kMaxRowBlocksKLo
                                          : kMaxRowBlocks;
  __shared__ uint16_t s_blk2[2][kRowBlocks];  // kv block list of this row / the next one
  // fp8: the k dequantisation scales of the listed blocks (read per tile: from global memory the
  // compiler would wait for every tile copy in flight along with them)
  __shared__ float s_ksc2[2][kFp8 ? kRowBlocks : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);  // wavefront index, kept scalar
  const int qs = wv & 3, kg = wv >> 2;
  const int l32 = lane & 31, g = lane >> 5;
  // The lane index, worked out again where it is called (two instructions) and opaque to the
  // compiler: address terms derived from the kernel-wide `lane` are computed once per launch, find no
  // register across the main loop and come back from scratch memory where they are used.
  auto fresh_lane = [&]() __attribute__((always_inline)) {
    int l = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    asm volatile("" : "+v"(l));
    return l;
  };
  const float c = p.sm_scale_log2;
  const TQK* __restrict__ qp = static_cast<const TQK*>(p.q);
  const TQK* __restrict__ kp = static_cast<const TQK*>(p.k);
  const T* __restrict__ vp = static_cast<const T*>(p.v);
  T* __restrict__ op = static_cast<T*>(p.o);
  uint8_t* const group_smem = smem + kg * kGroupBytes;

  // Copy assignment inside a kv group (4 wavefronts): copy instruction n = 4*j + qs, j = 0..3, fills
  // tile rows 4n..4n+3; this lane lands on row 4n + lane/16 at chunk position lane%16, so it must
  // fetch logical chunk (lane%16) ^ swz(row).  swz depends on row%16 = 4*qs + lane/16 only.
  const int cp_row = lane >> 4;
  const int cp_chunk = ((lane & 15) ^ swz(4 * qs + cp_row)) * 8;  // element offset inside the row
  // fp8 K tile (128-byte rows): copy instruction n = 4*j + qs, j = 0..1, fills rows 8n..8n+7; the
  // lane lands on row 8n + lane/8 at chunk position lane%8; swz8(row) = (4*(n%2) + lane/16) & 7
  const int cp8_row = lane >> 3;
  const int cp8_chunk = ((lane & 7) ^ ((4 * (qs & 1) + (lane >> 4)) & 7)) * 16;  // byte offset
  // K operand read: row mt*32 + l32, logical chunk 2*ks + g  ->  xor of a lane constant and ks<<5
  // (fp8: logical chunks 4*slab + 2*g and +1 of a 128-byte row)
  const int k_rd_base = l32 * (kFp8 ? kRowBytes8 : kRowBytes);
  const int k_rd_x = kFp8 ? ((2 * g) ^ swz8(l32)) << 4 : (g ^ swz(l32)) << 4;
  // V^T transpose read: this lane supplies row j = (lane%16)/4 of a 4-row patch that starts at kv
  // row 16*kk + 4*g (+8 for the second read), 8 bytes at element column 32*dt + 16*q2 + 4*(lane%4)
  int v_rd_off[4][2];
  if constexpr (!kPipe) {
    const int j = (lane & 15) >> 2, q2 = (lane >> 4) & 1, i4 = lane & 3;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int hi = 0; hi < 2; ++hi) {
        const int r = g * 4 + hi * 8 + j;
        const int chunk = dt * 4 + q2 * 2 + (i4 >> 1);
        v_rd_off[dt][hi] = r * kRowBytes + ((chunk ^ swz(r)) << 4) + (i4 & 1) * 8;
      }
  }

  // (what the widened form has left, most often nothing)
  if constexpr (kKLo)
    if (p.wide_left != nullptr && *p.wide_left == 0) return;
  // The next row is popped by kv group 1 while kv group 0 combines and stores the current one
  // (group 1 has nothing else to do then), so the queue atomics are off the critical path.
  if constexpr (!kDirect) {
    if (tid < kXcds) {
      const int lo = p.sched[tid], hi = p.sched[tid + 1];
      s_queue[tid] = lo;
      if (tid == kXcds - 1) s_queue[kXcds] = hi;
      s_behind[tid] = lo + static_cast<int>(gridDim.x + kXcds - 1 - tid) / kXcds;
      // (longest and shortest of eight lanes)
      int longest = hi - lo, shortest = longest;
      longest = max(longest, __builtin_amdgcn_update_dpp(longest, longest, 0xb1, 0xf, 0xf, false));  // quad_perm 1 0 3 2
      shortest = min(shortest, __builtin_amdgcn_update_dpp(shortest, shortest, 0xb1, 0xf, 0xf, false));
      longest = max(longest, __builtin_amdgcn_update_dpp(longest, longest, 0x4e, 0xf, 0xf, false));  // quad_perm 2 3 0 1
      shortest = min(shortest, __builtin_amdgcn_update_dpp(shortest, shortest, 0x4e, 0xf, 0xf, false));
      longest = max(longest, __builtin_amdgcn_update_dpp(longest, longest, 0x141, 0xf, 0xf, false));  // row_half_mirror
      shortest = min(shortest, __builtin_amdgcn_update_dpp(shortest, shortest, 0x141, 0xf, 0xf, false));
      if (tid == 0) {
        s_queue[kQueueUneven] = longest - shortest >= static_cast<int>(gridDim.x + kXcds - 1) / kXcds;
        s_guess = 0;  // (read first by a workgroup that is dealt no row)
      }
    }
    if (tid >= 64 && tid < 64 + 6) s_queue[9 + tid - 64] = p.sched[kSchedEven + tid - 64];
    __syncthreads();
  }
  // Even shares: the decoder has laid the rows out head by head and given every row a cost
  // (kRowOverhead + its kv blocks); share j is the cost range [j * share, (j + 1) * share), and a
  // row that straddles share boundaries is computed in parts by the shares it touches.  Every
  // workgroup holds one share; they are dealt so that the workgroups of one XCD hold neighbouring
  // shares (the same heads' K and V).  A share's items are consecutive rows of `order`, known from
  // the start: their records are gathered sixteen at a time, all in parallel, so that between two
  // rows only the kv block list has to be fetched.
  // (workgroup-uniform words: made scalar, so that none of them occupies a vector register for the
  // whole launch)
  auto queue_word = [&](int i) { return kDirect ? 0 : __builtin_amdgcn_readfirstlane(s_queue[i]); };
  const int ev_share = kDirect ? 1 : queue_word(10), ev_total = queue_word(11), ev_n = queue_word(12), ev_rows = queue_word(13);
  const bool even = kGroups == 2 && queue_word(9) != 0 && p.shares != nullptr && p.split_ws != nullptr &&
                    static_cast<int>(gridDim.x) == ev_n;
  const int ev_j = (ev_n & (kXcds - 1)) == 0 ? (blockIdx.x & (kXcds - 1)) * (ev_n / kXcds) + blockIdx.x / kXcds
                                             : static_cast<int>(blockIdx.x);
  auto fill_items = [&](int batch_base) {
    const int lane = fresh_lane();
    if (!kDirect && lane < kItemBatch) {
      RowInfo it;
      it.row = -1;
      it.ptr0 = 0;
      it.nb = 0;
      const int a = ev_j * ev_share, b = min(a + ev_share, ev_total);
      const int i = p.shares[ev_j] + batch_base + lane;
      const int32_t* row_start = p.shares + kMaxShares;
      if (a < ev_total && i < ev_rows) {
        const int u = row_start[i], e = row_start[i + 1] - kRowOverhead;  // kv blocks cost [u, e)
        // (a row without kv blocks stands for the last unit of its own overhead)
        if ((e > u ? u : u - 1) < b) {
          const int w = p.order[i];
          it.row = w;
          it.part = 0;
          it.parts = 1;
          it.slot = 0;
          if (e > u) {
            const int j_lo = u / ev_share, j_hi = (e - 1) / ev_share;
            it.part = ev_j - j_lo;
            it.parts = j_hi - j_lo + 1;
            it.slot = j_lo;
          }
          it.req = p.row_req[w];
          it.qb = p.row_qb[w];
          it.head = p.row_head[w];
          set_q_range(it, p.qo_indptr + it.req);
          it.kv_begin = p.kv_indptr[it.req];
          it.kv_len = p.kv_indptr[it.req + 1] - it.kv_begin;
          // this share's range of the row's kv blocks
          const int blk_lo = max(a, u) - u, blk_hi = min(min(b, e) - u, kRowBlocks);
          it.ptr0 = p.kv_row_ptr[w] + blk_lo;
          it.nb = max(blk_hi - blk_lo, 0);
          fill_scales(it);
        }
      }
      s_items[lane] = it;
    }
  };
  const bool have_records = queue_word(14) != 0 && p.shares != nullptr;
  int first_queue = 0;  // kept by the popping wavefront
  // One wavefront: lane 0 takes the next item (even shares: from the gathered records; otherwise it
  // pops a row and gathers its metadata, two rounds of loads), then all lanes copy the row's kv
  // block list; both go to LDS for the whole workgroup.
  auto fetch_next = [&](int slot_idx, bool dealt) {
    slot_idx = __builtin_amdgcn_readfirstlane(slot_idx);
    const int lane = fresh_lane();
    RowInfo ri;
    ri.row = -1;
    ri.ptr0 = 0;
    ri.nb = 0;
    if (even) {
      const int c = s_share[0];  // items handed out so far
      if (c > 0 && (c & (kItemBatch - 1)) == 0) fill_items(c);
      if (lane == 0) {
        ri = s_items[c & (kItemBatch - 1)];
        s_share[0] = c + 1;
        s_next_row[slot_idx] = ri;
      }
    } else {
      // Queues.  A workgroup's first row is the one of its XCD's queue at its own index (its record is asked
      // for straight away), the others are popped.  The trips to memory are kept to two: the pop's atomic
      // travels together with loads of the 64 records that follow this workgroup's last position in the
      // queue (the 32 workgroups of an XCD pop about once per row each, so the answer is nearly always one
      // of them; otherwise the record is read after the pop), and the row's bounds and its kv block list
      // are asked for together once the record is known.
      typedef __attribute__((ext_vector_type(4))) int i32x4;
      const int xcd = blockIdx.x & (kXcds - 1);
      const int own = queue_word(xcd) + static_cast<int>(blockIdx.x / kXcds);
      dealt = dealt && own < queue_word(xcd + 1);
      i32x4 w0 = {0, 0, 0, 0}, w1 = w0;  // lane i: the record at queue position win_lo + i
      int win_lo = 0, win_hi = 0;
      if (have_records) {
        const int fq = __builtin_amdgcn_readfirstlane(first_queue);
        if (fq < kXcds) {
          const int x = (xcd + fq) & (kXcds - 1);
          win_lo = dealt ? own : max(queue_word(x), __builtin_amdgcn_readfirstlane(s_guess));
          win_hi = min(queue_word(x + 1), win_lo + 64);
          if (win_lo + lane < win_hi) {
            const i32x4* rec = reinterpret_cast<const i32x4*>(p.shares + kMaxShares + kRecordInts * static_cast<int64_t>(win_lo + lane));
            w0 = rec[0];
            w1 = rec[1];
          }
        }
      }
      const int at = dealt ? own : pop_row(p, xcd, s_queue, s_behind, &first_queue, lane);
      ri.part = 0;
      ri.parts = 1;
      ri.slot = 0;
      if (at >= 0) {
        // (every lane forms the row's values: they are uniform, and lane 0 stores them)
        if (have_records) {
          i32x4 r0, r1;
          if (at >= win_lo && at < win_hi) {
            const int d = at - win_lo;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              r0[j] = __builtin_amdgcn_readlane(w0[j], d);
              r1[j] = __builtin_amdgcn_readlane(w1[j], d);
            }
          } else {
            const i32x4* rec = reinterpret_cast<const i32x4*>(p.shares + kMaxShares + kRecordInts * static_cast<int64_t>(at));
            r0 = rec[0];
            r1 = rec[1];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              r0[j] = __builtin_amdgcn_readfirstlane(r0[j]);
              r1[j] = __builtin_amdgcn_readfirstlane(r1[j]);
            }
          }
          ri.row = r0[0];
          ri.req = r0[1];
          ri.qb = r0[2];
          ri.head = r0[3];
          ri.ptr0 = r1[0];
          ri.nb = min(r1[1], kRowBlocks);
        } else {
          const int w = __builtin_amdgcn_readfirstlane(p.order[at]);
          ri.row = w;
          ri.req = __builtin_amdgcn_readfirstlane(p.row_req[w]);
          ri.qb = __builtin_amdgcn_readfirstlane(p.row_qb[w]);
          ri.head = __builtin_amdgcn_readfirstlane(p.row_head[w]);
          ri.ptr0 = __builtin_amdgcn_readfirstlane(p.kv_row_ptr[w]);
          // (a row longer than the LDS list is cut; the host side refuses such requests at plan time)
          ri.nb = min(__builtin_amdgcn_readfirstlane(p.kv_row_ptr[w + 1]) - ri.ptr0, kRowBlocks);
        }
        // the first 64 entries of the list are asked for before the bounds are waited for
        const int n = ri.nb, list0 = ri.ptr0;
        int blk_first = 0;
        if (lane < n) blk_first = p.kv_idx[list0 + lane];
        set_q_range(ri, p.qo_indptr + ri.req);
        ri.kv_begin = p.kv_indptr[ri.req];
        ri.kv_len = p.kv_indptr[ri.req + 1] - ri.kv_begin;
        fill_scales(ri);
        if (lane < n) {
          s_blk2[slot_idx][lane] = static_cast<uint16_t>(blk_first);
          if constexpr (kFp8) s_ksc2[slot_idx][lane] = p.k_scale[ri.k_scale0 + blk_first];
        }
        for (int i = 64 + lane; i < n; i += 64) {
          const int blk = p.kv_idx[list0 + i];
          s_blk2[slot_idx][i] = static_cast<uint16_t>(blk);
          if constexpr (kFp8) s_ksc2[slot_idx][i] = p.k_scale[ri.k_scale0 + blk];
        }
      }
      if (lane == 0) {
        s_next_row[slot_idx] = ri;
        s_guess = at + 1;
      }
    }
    if (even && __builtin_amdgcn_readfirstlane(ri.row) >= 0) {
      // (even shares: lane 0 holds the item; every lane copies its part of the kv block list)
      const int list0 = __builtin_amdgcn_readfirstlane(ri.ptr0), n = __builtin_amdgcn_readfirstlane(ri.nb);
      const int ks0 = __builtin_amdgcn_readfirstlane(ri.k_scale0);
      for (int i = lane; i < n; i += 64) {
        const int blk = p.kv_idx[list0 + i];
        s_blk2[slot_idx][i] = static_cast<uint16_t>(blk);
        if constexpr (kFp8) s_ksc2[slot_idx][i] = p.k_scale[ks0 + blk];
      }
    }
    // (everything fetched has been used; said explicitly so that the compiler does not carry these
    // loads as pending to the top of the row loop and wait there, behind the previous row's stores)
    __builtin_amdgcn_s_waitcnt(0x0f70);
  };
  // ---- kDirect: rows straight from the packed symbols (short lists) ----
  // Every workgroup reads all flags and keep bits itself, two, four, seven or eight candidates (symbol row, head) per
  // thread in head-major order, and works out with two or three workgroup scans which rows or parts of rows
  // are its own.  A decode launch in front of this one costs 8-15 us and a launch gap at these sizes, most of
  // it latency of a single workgroup; here the same trips to memory (two, for a batch of one request) replace
  // the three that fetching the decoded schedule costs.
  //   * Whole parts: one workgroup per row, or per part of it where workgroups are left over and a part still
  //     has kDirectMinPart kv blocks.  Where there are no more rows than workgroups and the longest part is
  //     no longer than an even share and what its cuts cost.
  //   * Even shares as the decoder lays them out (a row costs kShareRowCost + its kv blocks, a share is a range
  //     of that cost), with the table of the share's rows in LDS.  (154 rows of 260 kv blocks on 256 workgroups: 517 us as
  //     whole rows, 338 in shares; 160 rows of 64 blocks 139 -> 92.)
  // In the pipelined form the next item is fetched beside a row's first copies instead of at its end, where the
  // trips to memory are 2.4 us that nothing hides.
  __shared__ int s_wave[6][8];
  // even shares: the rows of this workgroup's share, where there may be more than the table holds row i at i % kDirectShareRows
  __shared__ uint16_t s_row_cand[kDirect ? kDirectShareRows : 1];  // a row's candidate ...
  __shared__ int s_row_u[kDirect ? kDirectShareRows + 1 : 1];      // ... and the cost at which its kv blocks begin
  auto row_at = [](int i) { return kMany != 0 ? i & (kDirectShareRows - 1) : i; };
  constexpr int kMaxCand = direct_max_cand(kMany);
  __shared__ uint16_t s_zero[kDirect ? kMaxCand / 16 : 1];         // candidates this workgroup clears (of 16 or more)
  // first row of the share, candidates to clear; even shares: the row behind its last one (0: one item at most), shares, cost of all,
  // the share's bounds
  // (in LDS and not in registers, where they would live through the main loop)
  __shared__ int s_dir[7];
  __shared__ int s_list_at;  // whole parts: where the item's keep bits are in LDS (words from smem on), or -1
  __shared__ int s_map[2];   // the piece of keep bits in the tile buffers until the first row: first word (as in DirectMask), words
  // even shares, pipelined form: keep bits of the items at hand, where they are no more than this (fetched with the items: a list that is made
  // beside a row's first copies must not wait for a load, which comes back behind them)
  constexpr int kBitWords = 34;
  __shared__ uint32_t s_bits[kDirect && kPipe ? kItemBatch : 1][kBitWords];
  __shared__ int s_ends[5];  // a batch of one request: its q and kv tokens, where its keep bits begin
  const uint8_t* const kv_info_words = kDirect && p.kv_info ? p.kv_info - (reinterpret_cast<uintptr_t>(p.kv_info) & 3) : nullptr;
  // this workgroup's share: neighbouring ones on one XCD
  auto dir_index = [&]() {
    return (gridDim.x & (kXcds - 1)) == 0 ? (blockIdx.x & (kXcds - 1)) * (gridDim.x / kXcds) + blockIdx.x / kXcds
                                          : static_cast<int>(blockIdx.x);
  };
  // floor(a / d) for a < 2^21: with half a unit added the quotient is further from a whole number than the
  // reciprocal's error
  auto part_of = [](int a, int d) {
    return static_cast<int>((static_cast<float>(a) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(d)));
  };
  // Share j of `shares` begins at cost cut_at(j) (products below 2^30: at most 2^20 keep bits, 512 shares).  Where two workgroups share a CU the one that was launched
  // first is ahead of the other throughout (its wavefronts are older and go first: 126.0 against 130.9 us with equal
  // shares, and the younger one then runs alone on its CU, at two thirds of the pair's rate), so the shares of an
  // XCD's first half are longer by kOlderGain / 128 and those of the second half shorter: ends at 121.4 and 122.3 us.
  // (Before the MFMAs of S had priority, whichever workgroup they are of, 126 and 146 us, and 10 / 128 was the best.)
  auto cut_at = [&](int j, int total, int shares) __attribute__((always_inline)) {
    if constexpr (kPipe) {
      const int per = shares / kXcds;
      if (shares == static_cast<int>(gridDim.x) && per * kXcds == shares && (per & 1) == 0) {
        const int i = j - part_of(j, per) * per;
        // 2^16 times the part of all cost that lies in front of share j
        const uint32_t in_front = static_cast<uint32_t>(j * 128 + min(i, per - i) * kOlderGain) * 512u / shares;
        return static_cast<int>((static_cast<uint64_t>(total) * in_front) >> 16);
      }
    }
    return static_cast<int>(static_cast<uint32_t>(j) * total / shares);
  };
  // everything about candidate `cand` but its part
  auto direct_row = [&](int cand, RowInfo& it) __attribute__((always_inline)) {
    const int h = part_of(cand, p.n_blk), t = cand - h * p.n_blk;
    it.row = cand;
    it.req = p.batch == 1 ? 0 : p.blk_req[t];
    it.qb = p.batch == 1 ? t : p.blk_qb[t];
    it.head = h;
    // (one request: its bounds are in LDS)
    const bool one = p.batch == 1;
    set_q_range(it, one ? s_ends : p.qo_indptr + it.req);
    it.kv_begin = one ? s_ends[2] : p.kv_indptr[it.req];
    it.kv_len = (one ? s_ends[3] : p.kv_indptr[it.req + 1]) - it.kv_begin;
    if constexpr (kDirect) {
      it.nkv = (it.kv_len + kBlockKV - 1) / kBlockKV;
      it.mask = 0;
      it.mask_first = 0;
      if (!p.is_full) {
        const BitRange r(p.kv_info + (one ? s_ends[4] : p.kv_info_indptr[it.req]),
                         static_cast<uint32_t>(it.qb * p.symbol_heads + h) * it.nkv, it.nkv);
        it.mask = static_cast<int>(r.words - reinterpret_cast<const uint32_t*>(kv_info_words));
        it.mask_first = r.first;
      }
    }
    it.q_scale = 1.f;
    it.k_scale0 = 0;
  };
  constexpr int kCands = (kMaxCand + 64 * kWaves - 1) / (64 * kWaves);  // candidates of a thread, at most
  auto direct_schedule = [&]() {
    const int n_wg = gridDim.x, n_cand = p.n_blk * p.symbol_heads, dir_g = dir_index();
    // (All of a thread's candidates, also where it does not have as many: with a branch around each of those, their loads are
    // waited for one after the other and their instructions do not mix.  9000 tokens x 8 heads over 500 29.6 -> 29.1 us, 808
    // candidates of five requests 36.7 -> 35.7, 6600 x 24 53.6 -> 51.4; 6 candidates 14.9 either way.)
    const int first_cand = kCands * tid;
    if (tid < kItemBatch) s_items[tid].row = -1;
    if (tid == 0) s_next_row[0].row = -1;
    // What this costs is instructions: every wavefront goes through all of it, and 2300 of them are 5 us.
    int list_at[kCands];  // where a candidate's keep bits are in LDS (words from smem on), or -1
    bool act[kCands];
    int n[kCands], map_word = 0, map_words = 0;
    const bool one = p.batch == 1;
    {
      // All of a thread's candidates make their trips to memory together: request, where it begins, flags and keep bits.
      // The keep bits come as one piece into the tile buffers, which nothing uses yet, where they fit.
      int req[kCands], bit[kCands], nkv[kCands];
      const int cand0 = min(first_cand, n_cand - 1);
      int h = part_of(cand0, p.n_blk), t = cand0 - h * p.n_blk;
#pragma unroll
      for (int u = 0; u < kCands; ++u) {
        req[u] = one ? 0 : p.blk_req[t];
        bit[u] = (one ? t : p.blk_qb[t]) * p.symbol_heads + h;
        act[u] = first_cand + u < n_cand;
        // (the next one, head by head; behind the last the last head again)
        const bool wrap = ++t == p.n_blk;
        t = wrap ? 0 : t;
        h = wrap ? min(h + 1, p.symbol_heads - 1) : h;
      }
      int ends[5] = {0, 0, 0, 0, 0}, map_lo = 0, map_hi = 0, info_at = 0;
      if (!p.is_full) {
        map_lo = p.kv_info_indptr[0];
        map_hi = p.kv_info_indptr[p.batch];
        info_at = p.info_indptr[0];
      }
      if (one) {
        ends[0] = p.qo_indptr[0];
        ends[1] = p.qo_indptr[1];
        ends[2] = p.kv_indptr[0];
        ends[3] = p.kv_indptr[1];
        ends[4] = map_lo;
#pragma unroll
        for (int u = 0; u < kCands; ++u) nkv[u] = (ends[3] - ends[2] + kBlockKV - 1) / kBlockKV;
      } else {
#pragma unroll
        for (int u = 0; u < kCands; ++u)
          nkv[u] = (p.kv_indptr[req[u] + 1] - p.kv_indptr[req[u]] + kBlockKV - 1) / kBlockKV;
      }
      if (p.is_full) {
#pragma unroll
        for (int u = 0; u < kCands; ++u) n[u] = act[u] ? nkv[u] : 0;
        if (one && tid == 0)
#pragma unroll
          for (int i = 0; i < 5; ++i) s_ends[i] = ends[i];
      } else {
        int keep_at[kCands];
        uint8_t flags[kCands];
        if (one) {
          const uint8_t* const info = p.info + info_at;
#pragma unroll
          for (int u = 0; u < kCands; ++u) {
            keep_at[u] = ends[4];
            flags[u] = info[bit[u] >> 3];
          }
        } else {
#pragma unroll
          for (int u = 0; u < kCands; ++u) {
            keep_at[u] = p.kv_info_indptr[req[u]];
            flags[u] = p.info[p.info_indptr[req[u]] + (bit[u] >> 3)];
          }
        }
        // (The indptr's last entry says where the segments end, and nothing else reads it: no further than the buffer, whose size a
        // launch that keeps a copy knows anyway.  A field of its own for it, one more word of kernel arguments, is 0.2 us of a
        // launch of 6 to 30.)
        const int map_bytes = min(map_hi, p.kv_info_bytes) - map_lo;
        const uint8_t* const at = p.kv_info + map_lo;
        const int skew = static_cast<int>(reinterpret_cast<uintptr_t>(at) & 3);
        const bool staged = map_bytes <= kDirectMapBytes;
        if (staged) {
          const uint32_t* src = reinterpret_cast<const uint32_t*>(at - skew);
          const int n_words = (skew + map_bytes + 3) >> 2;
          map_word = static_cast<int>(src - reinterpret_cast<const uint32_t*>(kv_info_words));
          map_words = n_words;
          uint32_t* dst = reinterpret_cast<uint32_t*>(smem);
          for (int i = tid; i < n_words; i += 4 * 64 * kWaves) {
            uint32_t v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = src[min(i + j * 64 * kWaves, n_words - 1)];
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (i + j * 64 * kWaves < n_words) dst[i + j * 64 * kWaves] = v[j];
          }
        }
        if (one && tid == 0)
#pragma unroll
          for (int i = 0; i < 5; ++i) s_ends[i] = ends[i];
        __syncthreads();
        int first[kCands], left = 0;
        bool beside = false;
#pragma unroll
        for (int u = 0; u < kCands; ++u) {
          act[u] = act[u] && (flags[u] >> (bit[u] & 7)) & 1;
          n[u] = 0;
          const uint32_t at_bit = static_cast<uint32_t>(bit[u]) * nkv[u];
          // (a caller's segments may lie in any order: one outside of the piece is read where it is)
          const bool inside = staged && keep_at[u] >= map_lo && keep_at[u] + static_cast<int>((at_bit + nkv[u] + 7) >> 3) <= map_lo + map_bytes;
          const int byte = skew + keep_at[u] - map_lo + static_cast<int>(at_bit >> 3);
          list_at[u] = inside ? byte >> 2 : -1;
          first[u] = (byte & 3) * 8 + static_cast<int>(at_bit & 7);
          if (act[u] && !inside) beside = true;
          if (act[u] && inside) left = max(left, nkv[u]);
        }
        if (beside) {
#pragma unroll
          for (int u = 0; u < kCands; ++u)
            if (act[u] && list_at[u] < 0) {
              const BitRange r(p.kv_info + keep_at[u], static_cast<uint32_t>(bit[u]) * nkv[u], nkv[u]);
              for (int i = 0; i < r.count(); ++i) n[u] += __popc(r.trim(r.words[i], i));
            }
        }
        // 32 kept blocks at a time (the word behind the last one is read as well: it is in the buffers, and masked)
        const uint32_t* words[kCands];
        uint32_t word[kCands];
#pragma unroll
        for (int u = 0; u < kCands; ++u) {
          nkv[u] = act[u] && list_at[u] >= 0 ? nkv[u] : 0;
          words[u] = reinterpret_cast<const uint32_t*>(smem) + max(list_at[u], 0);
          word[u] = words[u][0];
        }
        for (int i = 0; i < left; i += 32)
#pragma unroll
          for (int u = 0; u < kCands; ++u) {
            const uint32_t next = words[u][1];
            ++words[u];
            const int rest = max(nkv[u] - i, 0);
            uint32_t v = __builtin_amdgcn_alignbit(next, word[u], first[u]);
            v = rest >= 32 ? v : v & ~(~0u << rest);
            n[u] += __popc(v);
            word[u] = next;
          }
      }
    }
    if (tid < 3) s_dir[tid] = 0;
    // rows and kv blocks in one scan: at most 2047 and 2^20 of them
    constexpr int kBlockBits = 21;
    static_assert(kDirectMost < (1 << (32 - kBlockBits)), "rows must fit above the kv blocks");
    uint32_t mine = 0;
    int mx = 0;
#pragma unroll
    for (int u = 0; u < kCands; ++u) {
      mine += (static_cast<uint32_t>(act[u]) << kBlockBits) + n[u];
      mx = max(mx, n[u]);
    }
    const uint32_t incl = static_cast<uint32_t>(wave_scan(static_cast<int>(mine)));
    mx = wave_max(mx);
    if (lane == 63) {
      s_wave[0][wv] = static_cast<int>(incl);
      s_wave[2][wv] = mx;
    }
    __syncthreads();
    uint32_t all = 0, in_front = incl - mine;
    int max_n = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t t = static_cast<uint32_t>(s_wave[0][w]);
      if (w < wv) in_front += t;
      all += t;
      max_n = max(max_n, s_wave[2][w]);
    }
    all = __builtin_amdgcn_readfirstlane(all);
    max_n = __builtin_amdgcn_readfirstlane(max_n);
    const int rows = static_cast<int>(all >> kBlockBits), blocks = static_cast<int>(all & ((1u << kBlockBits) - 1));
    int row = static_cast<int>(in_front >> kBlockBits), before = static_cast<int>(in_front & ((1u << kBlockBits) - 1));
    // q blocks that are not computed are cleared by turns
    if (p.zero_skipped) {
      int skipped = first_cand - row;
#pragma unroll
      for (int u = 0; u < kCands; ++u)
        if (first_cand + u < n_cand && !act[u]) {
          const int turn = part_of(skipped, n_wg);
          if (skipped - turn * n_wg == dir_g) s_zero[turn] = static_cast<uint16_t>(first_cand + u);
          ++skipped;
        }
      if (tid == 0) s_dir[1] = max(n_cand - rows - dir_g + n_wg - 1, 0) / n_wg;
    }
    const int total = kShareRowCost * rows + blocks;
    // (a row in at most four parts: no share is shorter than a third of the longest row)
    int shares = max(min(n_wg, total), 1);
    if (3 * total < shares * max_n) shares = max(3 * total / max_n, 1);
    if (rows <= n_wg) {
      // Parts of at most `longest` kv blocks, as short as there are workgroups for.  Rows of n blocks make no more than n / longest
      // + 1 parts each, nor than the longest row does, and at least n / longest: where the two bounds leave a choice, the parts
      // are counted, two lengths at a time from the shortest on.  (Counted always, for every number of parts of the longest
      // row, with four scans, 108 rows of two requests took 1.3 us more.)
      const int finest = max(max((max_n + kDirectMaxParts - 1) / kDirectMaxParts, kDirectMinPart), part_of(blocks + n_wg - 1, n_wg));
      int longest = finest;
      if (rows * (part_of(max(max_n, 1) - 1, finest) + 1) > n_wg) {
        const int spare = n_wg - rows, per_row = max(part_of(n_wg, max(rows, 1)), 1);
        longest = max(finest, min(spare > 0 ? part_of(blocks + spare - 1, spare) : max_n, part_of(max_n + per_row - 1, per_row)));
      }
      for (int k = min(kDirectMaxParts, part_of(max_n + finest - 1, finest)), turn = 0; k > 0; k -= 2, turn ^= 1) {
        const int w0 = max(part_of(max_n + k - 1, k), finest), w1 = k > 1 ? max(part_of(max_n + k - 2, k - 1), finest) : w0;
        if (w0 >= longest) break;
        uint32_t parts_mine = 0;
#pragma unroll
        for (int u = 0; u < kCands; ++u) {
          const int last_block = max(n[u], 1) - 1;
          if (act[u]) parts_mine += static_cast<uint32_t>((part_of(last_block, w0) + 1) | (part_of(last_block, w1) + 1) << 16);
        }
        const int sum = wave_scan(static_cast<int>(parts_mine));
        if (lane == 63) s_wave[4 + turn][wv] = sum;
        __syncthreads();
        uint32_t parts_all = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) parts_all += static_cast<uint32_t>(s_wave[4 + turn][w]);
        parts_all = __builtin_amdgcn_readfirstlane(parts_all);
        if (static_cast<int>(parts_all & 0xffff) <= n_wg) {
          longest = w0;
          break;
        }
        if (static_cast<int>(parts_all >> 16) <= n_wg) {
          longest = min(longest, w1);
          break;
        }
      }
      // Whole parts or even shares: whichever has the least on its slowest workgroup.  A share is as good as never
      // made of one piece only: a second prologue, epilogue and exchange are worth kEvenExtra blocks.
      if (longest + (longest < max_n ? kPartExtra : 0) <= total / shares + kEvenExtra) {
        int parts[kCands], first = row;
#pragma unroll
        for (int u = 0; u < kCands; ++u) parts[u] = act[u];
        // (where no row is cut a part is a row, and the scan is left out: 6 candidates 15.5 -> 15.2 us; in the pipelined form,
        // whose four wavefronts are through with it sooner, the branch costs more than it saves: 808 candidates 36.4 -> 36.0 with it)
        if (kPipe || longest < max_n) {
          int parts_mine = 0;
#pragma unroll
          for (int u = 0; u < kCands; ++u) {
            parts[u] = act[u] ? part_of(max(n[u], 1) - 1, longest) + 1 : 0;
            parts_mine += parts[u];
          }
          const int parts_incl = wave_scan(parts_mine);
          if (lane == 63) s_wave[3][wv] = parts_incl;
          __syncthreads();
          first = parts_incl - parts_mine;
#pragma unroll
          for (int w = 0; w < kWaves; ++w)
            if (w < wv) first += s_wave[3][w];
        }
#pragma unroll
        for (int u = 0; u < kCands; ++u) {
          if (first <= dir_g && dir_g < first + parts[u]) {
            RowInfo it;
            direct_row(first_cand + u, it);
            const int per = (n[u] + parts[u] - 1) / parts[u];
            it.part = dir_g - first;
            it.parts = parts[u];
            it.slot = first;
            it.ptr0 = it.part * per;
            // (no part is empty but that of a row without kv blocks: per <= longest, so parts - 1 of them are fewer
            // than n blocks.  Longer than the LDS list, a part is cut, as the other forms cut a row: callers that
            // plan a batch send requests of more than kRowBlocks kv blocks to the decoder)
            it.nb = min(max(min(n[u] - it.ptr0, per), 0), kRowBlocks);
            s_next_row[0] = it;
            // its keep bits: in LDS already, or this thread's own
            s_list_at = p.is_full ? 0 : list_at[u];
          }
          first += parts[u];
        }
        __syncthreads();
        return;
      }
    }
    // Rows of the share alone: there are no more than the table holds (direct_table_holds).
    const int a = cut_at(dir_g, total, shares), b = cut_at(dir_g + 1, total, shares);
    int cost = kShareRowCost * row + before;
#pragma unroll
    for (int u = 0; u < kCands; ++u)
      if (act[u]) {
        const int after = cost + kShareRowCost + n[u];
        if (cost < b && a < after) {
          s_row_cand[row_at(row)] = static_cast<uint16_t>(first_cand + u);
          s_row_u[row_at(row)] = cost + kShareRowCost;
          // first row of the share: the one that holds the share's lower bound; its last one holds the upper bound's unit in front
          if (cost <= a) s_dir[0] = row;
          if (b <= after) {
            s_row_u[row_at(row + 1)] = after + kShareRowCost;
            s_dir[2] = row + 1;
          }
        }
        cost = after;
        ++row;
      }
    if (tid == 0) {
      s_map[0] = map_word;
      s_map[1] = map_words;
      if (dir_g >= shares) s_dir[2] = 1;  // (no row: see direct_items)
      s_dir[3] = shares;
      s_dir[4] = total;
      s_dir[5] = a;
      s_dir[6] = b;
    }
    __syncthreads();
  };
  // sixteen items of the share from `batch_base` on
  auto direct_items = [&](int batch_base) __attribute__((always_inline)) {
    const int lane = fresh_lane();
    if (lane < kItemBatch) {
      RowInfo it;
      it.row = -1;
      const int dir_g = dir_index(), rows = s_dir[2], shares = s_dir[3], total = s_dir[4];
      const int a = s_dir[5], b = s_dir[6], i = s_dir[0] + batch_base + lane;
      if (dir_g < shares && i >= 0 && i < rows) {
        // kv blocks cost [u, e)
        const int u = s_row_u[row_at(i)], e = s_row_u[row_at(i + 1)] - kShareRowCost;
        // (a row without kv blocks stands for the last unit of its own overhead)
        if ((e > u ? u : u - 1) < b) {
          direct_row(s_row_cand[row_at(i)], it);
          it.part = 0;
          it.parts = 1;
          it.slot = 0;
          if (e > u) {
            // (the shares that hold its first and its last kv block: this one, or some next to it)
            int j_lo = dir_g, j_hi = dir_g;
            if (u < a)
              do --j_lo; while (cut_at(j_lo, total, shares) > u);
            if (e > b)
              do ++j_hi; while (cut_at(j_hi + 1, total, shares) < e);
            it.part = dir_g - j_lo;
            it.parts = j_hi - j_lo + 1;
            it.slot = j_lo;
          }
          it.ptr0 = max(a, u) - u;
          it.nb = min(max(min(b, e) - u - it.ptr0, 0), kRowBlocks);
        }
      }
      s_items[lane] = it;
    }
    if constexpr (kDirect && kPipe) {
      if (p.is_full) return;
      // (four lanes to an item)
      const int k = lane & (kItemBatch - 1);
      const RowInfo& it = s_items[k];
      const int words = (it.mask_first + it.nkv + 31) >> 5;
      if (it.row >= 0 && words <= kBitWords) {
        const int in_map = it.mask - s_map[0];
        // (behind the first sixteen items the tile buffers are in use)
        if (batch_base == 0 && in_map >= 0 && in_map + words <= s_map[1]) {
          for (int i = lane >> 4; i < words; i += 4) s_bits[k][i] = reinterpret_cast<const uint32_t*>(smem)[in_map + i];
        } else {
          for (int i = lane >> 4; i < words; i += 4) s_bits[k][i] = reinterpret_cast<const uint32_t*>(kv_info_words)[it.mask + i];
        }
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);  // (see fetch_next)
    }
  };
  // One wavefront: the kv block list of the item in s_next_row[slot_idx], from the row's keep bits (words_at: in LDS from
  // there on, -1: in s_bits, row `bits_row`, or in memory)
  auto direct_list = [&](int slot_idx, const RowInfo& it, int words_at, int bits_row) __attribute__((always_inline)) {
    const int lane = fresh_lane();
    const int lo = __builtin_amdgcn_readfirstlane(it.ptr0), n = __builtin_amdgcn_readfirstlane(it.nb);
    if (p.is_full) {
      for (int i = lane; i < n; i += 64) s_blk2[slot_idx][i] = static_cast<uint16_t>(lo + i);
    } else if constexpr (kDirect) {
      BitRange r(nullptr, 0, __builtin_amdgcn_readfirstlane(it.nkv));
      r.first = __builtin_amdgcn_readfirstlane(it.mask_first);
      // a kv block per lane, its place in the list from the bits below it
      int seen = -lo;
      auto keep_bits = [&](int b, uint32_t word) __attribute__((always_inline)) {
        const bool kept = b < r.n && (word >> ((r.first + b) & 31)) & 1;
        const uint64_t all = __ballot(kept);
        const int at_bit = seen + static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(all >> 32),
                                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(all), 0u)));
        if (kept && at_bit >= 0 && at_bit < n) s_blk2[slot_idx][at_bit] = static_cast<uint16_t>(b);
        seen += __popcll(all);
      };
      if (words_at >= 0) {
        const uint32_t* const words = reinterpret_cast<const uint32_t*>(smem) + words_at;
        for (int b0 = 0; b0 < r.n && seen < n; b0 += 64) keep_bits(b0 + lane, words[(r.first + min(b0 + lane, r.n - 1)) >> 5]);
      } else if (kPipe && bits_row >= 0 && r.count() <= kBitWords) {
        const uint32_t* const words = s_bits[bits_row];
        for (int b0 = 0; b0 < r.n && seen < n; b0 += 64) keep_bits(b0 + lane, words[(r.first + min(b0 + lane, r.n - 1)) >> 5]);
      } else {
        r.words = reinterpret_cast<const uint32_t*>(kv_info_words) + __builtin_amdgcn_readfirstlane(it.mask);
        // four rounds' words requested together
        for (int b0 = 0; b0 < r.n && seen < n; b0 += 4 * 64) {
          uint32_t v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = r.words[(r.first + min(b0 + 64 * j + lane, r.n - 1)) >> 5];
#pragma unroll
          for (int j = 0; j < 4; ++j) keep_bits(b0 + 64 * j + lane, v[j]);
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);  // (see fetch_next)
      }
    }
  };
  // One wavefront: the next item and its list
  auto direct_next = [&](int slot_idx) __attribute__((always_inline)) {
    slot_idx = __builtin_amdgcn_readfirstlane(slot_idx);
    const int lane = fresh_lane();
    const int at = __builtin_amdgcn_readfirstlane(s_share[0]);  // items handed out so far
    if (at > 0 && (at & (kItemBatch - 1)) == 0) direct_items(at);
    const RowInfo& it = s_items[at & (kItemBatch - 1)];
    if (lane == 0) {
      s_next_row[slot_idx] = it;
      s_share[0] = at + 1;
    }
    if (__builtin_amdgcn_readfirstlane(it.row) >= 0) direct_list(slot_idx, it, -1, at & (kItemBatch - 1));
  };
  if constexpr (kDirect) {
    // The copy of the symbols for a later decode: 2 KB or so by each of the last workgroups, asked for in front of the
    // schedule and stored behind it.  (By all of them, with nothing between load and store, it was 0.6 us that every workgroup
    // waited; at the launch's end the last ones were 0.3 us late for it.)
    constexpr int kKeep = 4, kAll = 64 * kWaves;
    const int back = static_cast<int>(gridDim.x - 1 - blockIdx.x), keep_at = back * kKeep * kAll + tid, keep_ip = back * kAll + tid;
    const bool keeps = p.keep_info != nullptr && (back * kKeep * kAll < max(p.kv_info_bytes, p.info_bytes) || back * kAll <= p.batch);
    uint8_t kept_kv[kKeep], kept[kKeep];
    int32_t kept_ip[2];
    if (keeps) {
#pragma unroll
      for (int j = 0; j < kKeep; ++j) {
        const int i = keep_at + j * kAll;
        if (i < p.kv_info_bytes) kept_kv[j] = p.kv_info[i];
        if (i < p.info_bytes) kept[j] = p.info[i];
      }
      if (keep_ip <= p.batch) {
        kept_ip[0] = p.info_indptr[keep_ip];
        kept_ip[1] = p.kv_info_indptr[keep_ip];
      }
    }
    // (by the workgroup with the last share, which has the least to do: the first one is 0.4 us late for it, 1 % of
    // a launch of 33 us)
    if (p.keep_indptr != nullptr && blockIdx.x == gridDim.x - 1 && tid == 0) p.sched[kSchedKept] = p.is_full ? 2 : 1;
    direct_schedule();
    if (keeps) {
#pragma unroll
      for (int j = 0; j < kKeep; ++j) {
        const int i = keep_at + j * kAll;
        if (i < p.kv_info_bytes) p.keep_kv_info[i] = kept_kv[j];
        if (i < p.info_bytes) p.keep_info[i] = kept[j];
      }
      if (keep_ip <= p.batch) {
        p.keep_indptr[keep_ip] = kept_ip[0];
        p.keep_indptr[p.batch + 1 + keep_ip] = kept_ip[1];
      }
      // (more than the workgroups take at a time)
      const int all = static_cast<int>(gridDim.x) * kAll;
      for (int i = kKeep * all + back * kAll + tid; i < max(p.kv_info_bytes, p.info_bytes); i += all) {
        if (i < p.kv_info_bytes) p.keep_kv_info[i] = p.kv_info[i];
        if (i < p.info_bytes) p.keep_info[i] = p.info[i];
      }
      for (int i = all + keep_ip; i <= p.batch; i += all) {
        p.keep_indptr[i] = p.info_indptr[i];
        p.keep_indptr[p.batch + 1 + i] = p.kv_info_indptr[i];
      }
    }
    if (wv == 0) {
      if (lane == 0) s_share[0] = 0;
      if (__builtin_amdgcn_readfirstlane(s_dir[2]) > 0) {
        direct_items(0);
        direct_next(0);
      } else {
        // whole parts: the item is there, and the only one
        if (lane == 0) s_share[0] = 1;
        if (__builtin_amdgcn_readfirstlane(s_next_row[0].row) >= 0)
          direct_list(0, s_next_row[0], __builtin_amdgcn_readfirstlane(s_list_at), -1);
      }
    }
  }
  if constexpr (!kDirect) {
    if (wv == 0) {
      if (even) {
        if (lane == 0) s_share[0] = 0;
        fill_items(0);
      }
      fetch_next(0, true);
    }
  }
  for (int row_it = 0;; ++row_it) {
    // s_next_row is published; everyone is done with the previous row's LDS data.  (Not
    // __syncthreads(): its fence would also wait for the row just stored to be acknowledged by
    // memory, a few microseconds that nothing here depends on.)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const RowInfo& ri = s_next_row[row_it & 1];
    const int w = __builtin_amdgcn_readfirstlane(ri.row);  // uniform values, kept in scalar registers
    if (w < 0) break;
    const int part = __builtin_amdgcn_readfirstlane(ri.part), parts = __builtin_amdgcn_readfirstlane(ri.parts);
    const int split_slot = __builtin_amdgcn_readfirstlane(ri.slot);
    const int req = __builtin_amdgcn_readfirstlane(ri.req), qb = __builtin_amdgcn_readfirstlane(ri.qb);
    const int head = __builtin_amdgcn_readfirstlane(ri.head);
    const int q_begin = __builtin_amdgcn_readfirstlane(ri.q_begin);
    const int q_rows = __builtin_amdgcn_readfirstlane(ri.q_rows);
    const int kv_begin = __builtin_amdgcn_readfirstlane(ri.kv_begin);
    const int kv_len = __builtin_amdgcn_readfirstlane(ri.kv_len);
    const int nb = __builtin_amdgcn_readfirstlane(ri.nb);
    const uint16_t* const s_blk = s_blk2[row_it & 1];

    // (the lane's q row, from a lane index worked out here: see fresh_lane)
    const int lane_p = fresh_lane();
    const int l32_p = lane_p & 31, g_p = lane_p >> 5;
    const int my_row = qs * 32 + l32_p;  // q row of this lane inside the block
    const bool row_ok = my_row < q_rows;
    // row r of the item -> its token (relative to q_begin) and q head (relative to head_q0)
    // (a compile-time variant: as a run-time branch the mapping cost the ungrouped kernel 7 % at the
    // FLUX shape, in how the compiler arranged the code around it)
    const int gq = kGqaPack ? p.gqa_pack : 0;
    const int head_q0 = gq ? head * gq : head;
    auto row_at = [&](int r, int& tok, int& hq) __attribute__((always_inline)) {
      if constexpr (kGqaPack) {
        const uint32_t pr = static_cast<uint32_t>(qb) * kBlockQ + r;
        tok = static_cast<int>(pr / static_cast<uint32_t>(gq));
        hq = static_cast<int>(pr - tok * gq);
      } else {
        tok = r;
        hq = 0;
      }
    };
    // element offset of row r from the item's first q (o) vector, whose strides are sn, sh
    auto row_off = [&](int r, int64_t sn, int64_t sh) __attribute__((always_inline)) {
      int tok, hq;
      row_at(r, tok, hq);
      return tok * sn + hq * sh;
    };
    int my_tok, my_hq;
    row_at(row_ok ? my_row : q_rows - 1, my_tok, my_hq);
    const int64_t q_tok = q_begin + my_tok;
    const int my_head = head_q0 + my_hq;

    // one of the two forms of a call with widened operands takes this row
    bool other_form = false;
    if constexpr (kWide) {
      other_form = !wide_holds(ri.q_scale, p.wide_range[head / p.kv_group], c);
      if (other_form && tid == 0) *p.wide_left = 1;
    } else if constexpr (kKLo) {
      if (p.wide_left != nullptr) other_form = wide_holds(ri.q_scale, p.wide_range[head / p.kv_group], c);
    }
    if (nb == 0 || other_form) {
      // listed row without kv blocks: zeros, lse = -5e4
      if (row_ok && kg == 0 && !other_form) {
        T* dst = op + q_tok * p.o_sn + static_cast<int64_t>(my_head) * p.o_sh + g_p * 64;
        const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < 8; ++j) reinterpret_cast<u32x4*>(dst)[j] = z;
        if (p.lse && g_p == 0) p.lse[q_tok * p.num_heads + my_head] = kNegInf;
      }
      if (wv == kFetchWave) {
        if constexpr (kDirect) direct_next((row_it + 1) & 1); else fetch_next((row_it + 1) & 1, false);
      }
      continue;
    }

    f32x16 o_acc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o_acc[dt][i] = 0.f;
    float m_run = 0.f, d_part = 0.f;
    // kPipe: O^T as 16 x 16 tiles (16 d x 16 q rows), 2 * dt + qt: element j of a lane is d 16 * dt + 4 * (lane / 16) + j
    // of q row 16 * qt + lane % 16; reference point and row sum per q row (the sum over the lane's own keys)
    f32x4 o_tile[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) o_tile[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_q[2] = {0.f, 0.f}, d_q[2] = {0.f, 0.f};
    if constexpr (kPipe) {
      // ---- software-pipelined row (one kv group) ----
      // A step is 32 keys.  In step t a wavefront issues the MFMAs of S(t+1) = K(t+1).Q^T, sixteen tiles of 16 x 16 over 32 of
      // k, then the sixteen of O^T += V(t-1)^T.P(t-1)^T, and behind either run a part of the softmax of S(t) (exp2, rounding,
      // row sum -> P(t)); the largest value of S(t+1) is taken as soon as it is complete.  Eight operands are in registers,
      // each of two MFMAs: read eight operands ahead, into the registers of the one just used, V(t-1) during the MFMAs of S
      // and K(t+2) during those of P.V.  LDS holds four K and four V buffers of 32 keys; a copy is issued as soon as its
      // buffer is dead: K two and a half steps, V three before its first read.  One barrier per step.
      // What bounds it is the power limit and the vector ALU, which issues the MFMAs too: 32 of them, 16 exp2 and 26 other
      // instructions a step.  MFMA tiles of 32 x 32 over 16, half as many, read and write each accumulator twice as often and
      // held the clock at 1.55 GHz where these run at 1.8 (33 k tokens x 24 heads with windows, in 16 % fewer cycles at
      // equal interleaving).  What then made them the faster ones: K's swizzle (see q_chunk_of), and runs of MFMAs in place of
      // MFMAs and exponentials in turn, see the softmax's bursts.  33 k x 24 1782 -> 1700 us, 16 896 x 24 with a fifth of the
      // blocks in fp16 728 -> 693, 4608 x 24 from the symbols 115.9 -> 110.6, the layer step of 76 112 x 5120 with two-term
      // fp8 14 320 -> 14 002.
      constexpr int kStep = 32;
      // K buffers 0..2 | V buffer 0 | K buffer 3 | V buffers 1..3; Q is staged from K buffer 3 on, so
      // that K(0..2) and V(0) can be requested together with it
      constexpr int kQStage = 3 * kPipeKBuf + kPipeVBuf;
      static_assert(kPipeKBuf + 3 * kPipeVBuf >= kBlockQ * kRowBytes, "Q must fit behind K(0..2) and V(0)");
      auto kbuf = [&](int i) { return static_cast<uint32_t>(i * kPipeKBuf + (i == 3 ? kPipeVBuf : 0)); };
      auto vbuf = [&](int i) { return static_cast<uint32_t>((i == 0 ? 3 : 4) * kPipeKBuf + i * kPipeVBuf); };
      const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)smem));
      const int last_valid = min(kBlockKV, kv_len - s_blk[nb - 1] * kBlockKV);
      const int n_steps = 4 * (nb - 1) + ((last_valid + kStep - 1) / kStep);
      const int kv_head = head / p.kv_group;
      // (a widened k is laid out block by block, wherever the batch's tokens begin)
      const uint8_t* k_head = reinterpret_cast<const uint8_t*>(
          kp + (kWide ? static_cast<int64_t>(__builtin_amdgcn_readfirstlane(ri.k_scale0)) * (kBlockKV * kHeadDim)
                      : static_cast<int64_t>(kv_begin) * p.k_sn + static_cast<int64_t>(kv_head) * p.k_sh));
      const uint8_t* v_head = reinterpret_cast<const uint8_t*>(
          vp + static_cast<int64_t>(kv_begin) * p.v_sn + static_cast<int64_t>(kv_head) * p.v_sh);
      // K and V copies go through buffer descriptors that end with the request's last key: a copy
      // that reaches past it (the ragged last 32 keys, or the copies a row's last steps issue for steps
      // that do not exist) touches no memory there, so the loop issues its copies unconditionally.
      // Offsets are 32 bits: the launcher picks this kernel only for kv spans below 4 GiB.
      const uint32_t k_sn2 = static_cast<uint32_t>(p.k_sn) * sizeof(T), v_sn2 = static_cast<uint32_t>(p.v_sn) * sizeof(T);
      const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(k_head), 0, static_cast<uint32_t>(kv_len - 1) * k_sn2 + kRowBytes, 0x00020000);
      const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(v_head), 0, static_cast<uint32_t>(kv_len - 1) * v_sn2 + kRowBytes, 0x00020000);
      // A lane's part of a copy: row 4 * qs + lane / 16 of a 16-row group, 16-byte chunk swizzled.  (The operand reads of the
      // loop then differ by immediate offsets but for two bits of the chunk: four addresses each for K and V.)
      const int ln_c = fresh_lane();
      const int cp_chunk = (ln_c & 15) ^ ((ln_c >> 4) << 2), cp_row = 4 * qs + (ln_c >> 4);
      uint32_t k_voff = static_cast<uint32_t>(cp_row) * k_sn2 + (cp_chunk ^ qs) * 16;
      uint32_t v_voff = static_cast<uint32_t>(cp_row) * v_sn2 + cp_chunk * 16;
      asm volatile("" : "+v"(k_voff), "+v"(v_voff));
      // LDS addresses of this wavefront's part of buffer offset 0
      const uint32_t m0_k = lds0 + qs * 1024, m0_v = lds0 + qs * kPipeVRows4;
      // 64 lanes x 16 bytes of 4 rows, global -> LDS (see copy16_to_lds), addressed through a descriptor:
      // lane offset + scalar offset
      auto copy_desc = [&](__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff, uint32_t lds_addr) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
                     : "memory", "m0");
      };
      auto step_start = [&](int t) { return s_blk[t >> 2] * kBlockKV + (t & 3) * kStep; };
      // the 32 keys of step t (two copy instructions per wavefront) -> their LDS buffer
      auto copy_k = [&](int t) __attribute__((always_inline)) {
        const uint32_t soff = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(step_start(t))) * k_sn2;
#pragma unroll
        for (int j = 0; j < 2; ++j) copy_desc(k_rsrc, k_voff, soff + j * 16 * k_sn2, m0_k + kbuf(t & 3) + j * 4096);
      };
      auto copy_v = [&](int t) __attribute__((always_inline)) {
        const uint32_t soff = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(step_start(t))) * v_sn2;
#pragma unroll
        for (int j = 0; j < 2; ++j) copy_desc(v_rsrc, v_voff, soff + j * 16 * v_sn2, m0_v + vbuf(t & 3) + j * (4 * kPipeVRows4));
      };

      // prologue: Q, K(0..2), V(0) requested together
      if constexpr (kWide) {
        // (two tiles of 128-byte rows: q, then q_lo)
        const int ln_q = fresh_lane();
        const int q_row = ln_q >> 3, q_chunk = ((ln_q & 7) ^ ((4 * (qs & 1) + (ln_q >> 4)) & 7)) * 16;
        const int64_t q_off = static_cast<int64_t>(q_begin) * p.q_sn + static_cast<int64_t>(head_q0) * p.q_sh;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          int r = 8 * (4 * (n & 3) + qs) + q_row;
          r = r < q_rows ? r : q_rows - 1;
          copy16_to_lds(static_cast<const uint8_t*>(n < 4 ? p.q : p.q_lo) + q_off,
                        static_cast<uint32_t>(r * p.q_sn + q_chunk), lds0 + kQStage + qs * 1024 + n * 4096);
        }
      } else {
        const uint8_t* q_head = reinterpret_cast<const uint8_t*>(
            qp + static_cast<int64_t>(q_begin) * p.q_sn + static_cast<int64_t>(head_q0) * p.q_sh);
        const int ln_q = fresh_lane();
        const int cp_row = ln_q >> 4, cp_chunk = ((ln_q & 15) ^ swz(4 * qs + cp_row)) * 8;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          int r = 4 * (4 * n + qs) + cp_row;
          r = r < q_rows ? r : q_rows - 1;  // ragged last q block: re-read the last row
          copy16_to_lds(q_head, static_cast<uint32_t>((row_off(r, p.q_sn, p.q_sh) + cp_chunk) * sizeof(T)),
                        lds0 + kQStage + qs * 1024 + n * 4096);
        }
      }
      copy_k(0);
      if (n_steps > 1) copy_k(1);
      if (n_steps > 2) copy_k(2);
      copy_v(0);
      // Block numbers of the row's list as scalars: blk0 = the block of the current four steps, blk1
      // the one after it.  They come from a register that holds 64 consecutive entries of the list,
      // one per lane, refilled every 64 blocks: the loop itself reads no list from LDS (the wait
      // for such a read would also wait for the operand reads in flight).
      int blk_win = 0, blk0 = 0, blk1 = 0;
      // kWide: the factor that makes a logit of S, per kv block: softmax scale, q block's scale, k block's scale, in fp32
      // as in the fp8 form.  Kept like the block numbers; the first 64 are asked for beside the copies.
      float f_win = 0.f, f_blk = 1.f;
      auto k_factor = [&]() __attribute__((always_inline)) {
        return p.k_scale[__builtin_amdgcn_readfirstlane(ri.k_scale0) + blk_win];
      };
      if constexpr (kWide) {
        blk_win = s_blk[min(lane, nb - 1)];
        f_win = k_factor();
      }
      // (shares are known from the start: the next item and its kv block list are fetched beside these copies)
      if constexpr (kDirect)
        if (wv == 0) direct_next((row_it + 1) & 1);
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      __builtin_amdgcn_s_barrier();
      q8 qreg[8];  // 2 * ks + qt: 32 d of 16 q rows
      u32x4 op[8];  // operands of the next eight MFMAs: slices of K or of V^T
      u32x4 pA[2], pB[2];  // P of a step, per q tile: 8 rounded values, as 32-bit pairs
      f32x4 sA[4], sB[4];  // S of a step, 16 x 16 tiles 2 * kt + qt: keys 16 * kt + 4 * (lane / 16) + j of q row 16 * qt + lane % 16
      // Which 8 of an operand's 32 d a group of 16 lanes holds, of Q and of K alike: 0, 3, 1, 2.  A ds_read_b128 serves lanes 0-3
      // and 12-15 of a group together with lanes 4-11 of the next one; in this order, with K's swizzle, they meet in no bank
      // (in ascending order, as the counters have it, every read took twice as long).
      auto q_chunk_of = [](int ln) __attribute__((always_inline)) { return (0x9c >> (ln >> 4 << 1)) & 3; };
      if constexpr (kWide) {
        // q + q_lo in fp16 (the scales are applied to S)
        f_win *= c * ri.q_scale;
        const int ln_r = fresh_lane(), gr = q_chunk_of(ln_r);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int row = qs * 32 + (i & 1) * 16 + (ln_r & 15);
          const uint8_t* at = smem + kQStage + row * kRowBytes8 + (((i & ~1) + (gr >> 1)) ^ swz8(row)) * 16 + (gr & 1) * 8;
          const u32x2 hi = *reinterpret_cast<const u32x2*>(at), lo = *reinterpret_cast<const u32x2*>(at + 128 * kRowBytes8);
          widen8(hi, lo, qreg[i]);
        }
      } else {
        const int ln_r = fresh_lane();
        const int q_rd_base = (ln_r & 15) * kRowBytes, q_rd_x = (q_chunk_of(ln_r) ^ swz(ln_r & 15)) << 4;
        const uint8_t* qt = smem + kQStage + qs * 32 * kRowBytes + q_rd_base;
#pragma unroll
        for (int i = 0; i < 8; ++i) qreg[i] = *reinterpret_cast<const q8*>(qt + (i & 1) * 16 * kRowBytes + (q_rd_x ^ ((i >> 1) << 6)));
        // the softmax scale (log2 domain) is folded into Q, so S^T needs no multiply
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) qreg[i][e] = static_cast<T>(static_cast<float>(qreg[i][e]) * c);
      }
      // LDS addresses of the operand reads, without the buffer's offset and what else is an immediate of the read
      typedef __attribute__((address_space(3))) const q8 lds_x8;
      uint32_t krd[4], vrd[4];
      {
        const int ln = fresh_lane();
        const int r = ln & 15, j = r >> 2;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          krd[x] = lds0 + r * kRowBytes + ((x ^ (r & 3)) << 6) + ((q_chunk_of(ln) ^ (r >> 2)) << 4);
          // (row 4 * (lane / 16) + j, columns 32 * x + 4 * (lane % 4): see lds_read_tr16)
          vrd[x] = lds0 + (ln >> 4) * kPipeVRows4 + j * kRowBytes + ((x ^ j) << 6) + (ln & 3) * 8;
          asm volatile("" : "+v"(krd[x]), "+v"(vrd[x]));
        }
      }
      // K operand i = 2 * ks + kt (32 d of 16 keys) of the step whose K is in buffer `buf`
      auto read_k = [&](int buf, int i) __attribute__((always_inline)) {
        return *reinterpret_cast<lds_x8*>(static_cast<uintptr_t>(krd[i >> 1] + kbuf(buf) + (i & 1) * 4096));
      };
      // V^T operand dt of the step whose V is in buffer `buf`: 16 d x 32 keys, transposed; a lane's keys are those that it
      // has of S: 4 * (lane / 16) + 0..3, and 16 on
      auto read_v = [&](int buf, int dt) __attribute__((always_inline)) {
        union {
          s16x4 h[2];
          x8 v;
        } a;
        const uint32_t at = vrd[dt >> 1] + vbuf(buf) + (dt & 1) * 32;
        a.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(static_cast<uintptr_t>(at)));
        a.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_s16x4*>(static_cast<uintptr_t>(at + 4 * kPipeVRows4)));
        return a.v;
      };
#pragma unroll
      for (int e = 0; e < 4; ++e) sA[e] = f32x4{0.f, 0.f, 0.f, 0.f};
      {
        q8 k0[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) k0[i] = read_k(0, i);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int kt = (i >> 1) & 1, qt = i & 1, ks = i >> 2;
          sA[2 * kt + qt] = TS::mfma16(k0[2 * ks + kt], qreg[2 * ks + qt], sA[2 * kt + qt]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      // (a row of one step reads a buffer nobody filled: the result is never used)
#pragma unroll
      for (int i = 0; i < 8; ++i) op[i] = __builtin_bit_cast(u32x4, read_k(1, i));
      // (a row's first step multiplies P(-1) = 0 by what it reads from V buffer 3, where Q was staged: that must be
      // finite whatever Q holds)
#pragma unroll
      for (int e = 0; e < 4; ++e) pA[0][e] = pA[1][e] = pB[0][e] = pB[1][e] = 0u;
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): Q and K(0) are in registers
      __builtin_amdgcn_s_barrier();        // ... of every wavefront: their LDS space is free
      {
        // V buffer 3 (read by the first step as "V(-1)"), and for a row of fewer than four steps
        // every V buffer it does not fill (read by its padded steps), must not hold Q any more
        const u32x4 z = {0u, 0u, 0u, 0u};
        for (int b = min(n_steps, 3); b < 4; ++b) {
          uint8_t* vb = smem + vbuf(b) + wv * kPipeVRows4 + lane * 16;
          *reinterpret_cast<u32x4*>(vb) = z;
          *reinterpret_cast<u32x4*>(vb + 4 * kPipeVRows4) = z;
        }
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the zeros are there, before the barrier of the first step
      if (n_steps > 1) {
        copy_k(min(3, n_steps - 1));  // (kept to four instructions per group: the loop's waits count them)
        copy_v(1);
      }
      if constexpr (!kWide) blk_win = s_blk[min(lane, nb - 1)];
      typedef __attribute__((ext_vector_type(2))) T x2;
      const x2 ones2 = {static_cast<T>(1.0f), static_cast<T>(1.0f)};
      // keys of a step that a lane's half row does not have: p = 0
      auto mask_tail = [&](f32x4 (&s)[4], int valid) __attribute__((always_inline)) {
        const int g4 = (fresh_lane() >> 4) * 4;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i >> 2][i & 3] = (i >> 3) * 16 + (i & 3) + g4 < valid ? s[i >> 2][i & 3] : -INFINITY;
      };
      auto row_max = [&](const f32x4 (&s)[4], int qt) __attribute__((always_inline)) {
        float mx = s[qt][0];
#pragma unroll
        for (int i = 1; i < 8; ++i) mx = fmaxf(mx, s[qt + (i >> 2) * 2][i & 3]);
        return max_across_rows(max_across_halves(mx));
      };
      // What S accumulates from, per q tile: the reference point, taken off (kWide: nothing, it comes off with the factor).
      f32x4 s_init[2];
      const int valid0 = kv_len - static_cast<int>(s_blk[0]) * kBlockKV;
      if (valid0 < kStep) mask_tail(sA, valid0);
      const float s_max0[2] = {row_max(sA, 0), row_max(sA, 1)};
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        m_q[qt] = s_max0[qt];
        if constexpr (kWide) {
          m_q[qt] *= __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, f_win)));
          s_init[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
          asm volatile("" : "+v"(s_init[qt]));  // (held: as a constant it would be moves in every step)
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            sA[qt][j] -= m_q[qt];
            sA[2 + qt][j] -= m_q[qt];
            s_init[qt][j] = -m_q[qt];
          }
        }
      }
      // The largest S of the lane in the step at hand, of both its q rows.  As an integer (kWide: not, and per row), which is
      // right where any is positive, and the instruction does not quiet its operands first.
      using over_t = typename std::conditional<kWide, float, int>::type;
      over_t s_over[kWide ? 2 : 1] = {};
      if constexpr (kWide) {
        s_over[0] = s_max0[0];
        s_over[1] = s_max0[1];
      }
      // One step (kB = t % 4 picks the LDS buffers).  Straight-line code apart from small
      // wavefront-uniform branches, so that the accumulators stay where they are.
      auto do_step = [&](int t, auto buf_tag, f32x4 (&s_cur)[4], f32x4 (&s_next)[4], u32x4 (&p_prev)[2], u32x4 (&p_cur)[2]) __attribute__((always_inline)) {
        constexpr int kB = decltype(buf_tag)::value;
        // V(t-1) and K(t+2), first read in this step, have landed once only what was asked for after them is outstanding:
        // V(t) of step t-2 and the four copies of step t-1 (K goes first in every step); after the barrier that holds for
        // every wavefront.  The buffers that this step's copies overwrite, K(t)'s and V(t-2)'s, were last read in steps
        // t-2 and t-1, for MFMAs that every wavefront has issued by now.
        __builtin_amdgcn_s_waitcnt(0x0f70 | 6);  // vmcnt(6)
        __builtin_amdgcn_s_barrier();
        // This step's copies: K(t+4) and V(t+2).  Their scalar offsets are worked out here from the block numbers held
        // in scalar registers.  Steps past the row's end copy a block again or nothing (see the descriptors).
        const uint32_t v_soff = static_cast<uint32_t>(((kB + 2) < 4 ? blk0 : blk1) * kBlockKV + ((kB + 2) & 3) * kStep) * v_sn2;
        const uint32_t k_soff = static_cast<uint32_t>(blk1 * kBlockKV + kB * kStep) * k_sn2;
        // (a row is padded to a multiple of four steps; a padded step has no keys: p = 0, against V
        // operands read from buffers that hold earlier steps of the same row)
        const int valid = t < n_steps ? min(kStep, kv_len - (blk0 * kBlockKV + kB * kStep)) : 0;
        if (valid < kStep) mask_tail(s_cur, valid);
        // The reference point moves only past a 2^8 overshoot (a rare, wavefront-uniform branch that changes registers in
        // place): S(t), what S(t+1) accumulates from and the row sum move now; O, which still receives P(t-1).V(t-1) at
        // the old point in this step, is rescaled at the step's end.
        bool over;
        if constexpr (kWide) {
          over = __builtin_fmaf(s_over[0], f_blk, -m_q[0]) > kLazyLog2 || __builtin_fmaf(s_over[1], f_blk, -m_q[1]) > kLazyLog2;
        } else {
          over = s_over[0] > __builtin_bit_cast(int, kLazyLog2);
        }
        const bool moved = __builtin_expect(__any(over), 0);
        float o_scale[2] = {1.f, 1.f};
        if (moved) {
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) {
            float mx = row_max(s_cur, qt);  // row max relative to m_q
            if constexpr (kWide) mx = __builtin_fmaf(mx, f_blk, -m_q[qt]);
            const float delta = fmaxf(mx, 0.f);
            o_scale[qt] = __builtin_amdgcn_exp2f(-delta);
            d_q[qt] *= o_scale[qt];
            m_q[qt] += delta;
            if constexpr (!kWide) {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                s_cur[qt][j] -= delta;
                s_cur[2 + qt][j] -= delta;
                s_init[qt][j] -= delta;
              }
            }
          }
        }
        // The softmax of S(t) goes in two bursts, after the MFMAs of S(t+1) and after those of P.V: six exponentials and ten,
        // the first six's rounding and row sum (over the rounded values, as the reference takes it) in the second one, so
        // that nothing waits for the instruction in front of it.  An exponential takes the vector ALU as long as an MFMA the
        // matrix core; between two MFMAs of the same wavefront it delays the second one, behind a run of them the other
        // workgroup's wavefront has the matrix core.
        float psum[2] = {0.f, 0.f};
        float x[16];
        // value m of the lane's P: eight of q tile 0, then of q tile 1; of either four of keys 0..15, then of 16..31
        auto logit = [&](int m) __attribute__((always_inline)) {
          float f = s_cur[((m >> 2) & 1) * 2 + (m >> 3)][m & 3];
          if constexpr (kWide) {
            const float e = f;
            asm volatile("v_fma_f32 %0, %1, %2, -%3" : "=v"(f) : "v"(e), "s"(f_blk), "v"(m_q[m >> 3]));
          }
          return f;
        };
        // (Volatile, so that they stay where they are: the compiler gathers all exponentials of a step in front of its MFMAs
        // otherwise.  It does not see what they are, so the waits that they need are here: three states between an MFMA and a
        // write of what may have been its third operand, one between an exponential and whoever reads it.)
        auto exponentials = [&](int from, int to) __attribute__((always_inline)) {
          float f[16];
          asm volatile("s_nop 2");
#pragma unroll
          for (int m = from; m < to; ++m) f[m] = logit(m);
#pragma unroll
          for (int m = from; m < to; ++m) asm volatile("v_exp_f32 %0, %1" : "=v"(x[m]) : "v"(f[m]));
        };
        auto round_and_add = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
          for (int u = from / 2; u < to / 2; ++u) {
            const x2 pk = {static_cast<T>(x[2 * u]), static_cast<T>(x[2 * u + 1])};
            p_cur[u >> 2][u & 3] = __builtin_bit_cast(uint32_t, pk);
          }
#pragma unroll
          for (int u = from / 2; u < to / 2; ++u) {
            const x2 pk = __builtin_bit_cast(x2, static_cast<uint32_t>(p_cur[u >> 2][u & 3]));
            if constexpr (std::is_same<T, __bf16>::value) {
              psum[u >> 2] = __builtin_amdgcn_fdot2_f32_bf16(pk, ones2, psum[u >> 2], false);
            } else {
              psum[u >> 2] = __builtin_amdgcn_fdot2(pk, ones2, psum[u >> 2], false);
            }
          }
        };
        auto largest = [&](int from, int to) __attribute__((always_inline)) {
          auto bits = [&](int j) __attribute__((always_inline)) { return __builtin_bit_cast(over_t, static_cast<float>(s_next[j >> 2][j & 3])); };
          auto larger = [](over_t a, over_t b) __attribute__((always_inline)) {
            if constexpr (kWide) return fmaxf(a, b);
            else return max(a, b);
          };
#pragma unroll
          for (int j = from; j < to; ++j) {
            over_t& most = s_over[kWide ? (j >> 2) & 1 : 0];
            most = j == 0 || (kWide && j == 4) ? bits(j) : larger(most, bits(j));
          }
        };
        constexpr int kFirst = 6;  // (4 and 8: 0.3 and 1 % longer, 2 of 16: 5 %; in bursts of two 3 %, all sixteen at once 5 %)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < 16; ++n) {
          const int i = n & 7;
#pragma unroll
          for (int qt = 0; qt < 2; ++qt) {
            if (n < 8) {
              f32x4& to = s_next[2 * (i & 1) + qt];
              to = TS::mfma16(__builtin_bit_cast(q8, op[i]), qreg[2 * (i >> 1) + qt], n < 2 ? s_init[qt] : to);
            } else {
              o_tile[2 * i + qt] = TT::mfma16(__builtin_bit_cast(x8, op[i]), __builtin_bit_cast(x8, p_prev[qt]), o_tile[2 * i + qt]);
            }
          }
          if (n < 8) op[i] = __builtin_bit_cast(u32x4, read_v((kB + 3) & 3, i));
          else op[i] = __builtin_bit_cast(u32x4, read_k((kB + 2) & 3, i));
          __builtin_amdgcn_sched_barrier(0);
          if (n == 7) {
            exponentials(0, kFirst);
          } else if (n == 15) {
            round_and_add(0, kFirst);
            exponentials(kFirst, 16);
            asm volatile("s_nop 0" : "+v"(x[6]), "+v"(x[7]), "+v"(x[8]), "+v"(x[9]), "+v"(x[10]), "+v"(x[11]), "+v"(x[12]), "+v"(x[13]),
                                     "+v"(x[14]), "+v"(x[15]));
            round_and_add(kFirst, 16);
          }
          // (kWide, with two maxima: all of it at the end, 0.6 % of the layer's time)
          if (kWide && n == 15) largest(0, 16);
          if (!kWide && n >= 12) largest(n == 12 ? 0 : 4 * n - 49, 4 * n - 45 + (n == 15));
          // The MFMAs of P.V go first where the other workgroup's wavefront on this SIMD has some of S or softmax work ready:
          // 1742 -> 1714 us on the video-sized list; both kinds first 1778, softmax work after S as well 1750, nobody 1760.
          if (n == 7) __builtin_amdgcn_s_setprio(1);
          if (n == 15) __builtin_amdgcn_s_setprio(0);
          // (the copies of K among the MFMAs of S, those of V among P.V's: 1 % longer; all four at n = 7: 3 %)
          if (n == 1) copy_desc(k_rsrc, k_voff, k_soff, m0_k + kbuf(kB));
          if (n == 3) copy_desc(k_rsrc, k_voff, k_soff + 16 * k_sn2, m0_k + kbuf(kB) + 4096);
          if (n == 4) copy_desc(v_rsrc, v_voff, v_soff, m0_v + vbuf((kB + 2) & 3));
          if (n == 6) copy_desc(v_rsrc, v_voff, v_soff + 16 * v_sn2, m0_v + vbuf((kB + 2) & 3) + 4 * kPipeVRows4);
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("" : "+v"(psum[0]), "+v"(psum[1]), "+v"(p_cur[1][2]), "+v"(p_cur[1][3]), "+v"(s_over[0]));
        d_q[0] += psum[0];
        d_q[1] += psum[1];
        if (moved) {
#pragma unroll
          for (int e = 0; e < 16; ++e) o_tile[e] *= o_scale[e & 1];
        }
      };
      using B0 = std::integral_constant<int, 0>;
      using B1 = std::integral_constant<int, 1>;
      using B2 = std::integral_constant<int, 2>;
      using B3 = std::integral_constant<int, 3>;
      for (int t = 0; t < n_steps; t += 4) {
        const int bi = t >> 2;
        blk0 = __builtin_amdgcn_readlane(blk_win, bi & 63);
        if constexpr (kWide)
          f_blk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f_win), bi & 63));
        if (((bi + 1) & 63) == 0) {
          blk_win = s_blk[min(bi + 1 + lane, nb - 1)];
          if constexpr (kWide) f_win = c * ri.q_scale * k_factor();
        }
        blk1 = __builtin_amdgcn_readlane(blk_win, (bi + 1) & 63);
        do_step(t, B0{}, sA, sB, pB, pA);
        do_step(t + 1, B1{}, sB, sA, pA, pB);
        do_step(t + 2, B2{}, sA, sB, pB, pA);
        do_step(t + 3, B3{}, sB, sA, pA, pB);
      }
      __builtin_amdgcn_s_setprio(0);
      // P.V of the last step (real or padded; its V is in buffer 3)
      // (addresses that the compiler does not know to be the loop's: those that both use it would form ahead of the loop, in
      // sixteen registers, in place of immediate offsets)
#pragma unroll
      for (int x = 0; x < 4; ++x) asm volatile("" : "+v"(vrd[x]));
      __builtin_amdgcn_s_waitcnt(0x0f70 | 6);  // vmcnt(6)
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int i = 0; i < 8; ++i) op[i] = __builtin_bit_cast(u32x4, read_v(3, i));
#pragma unroll
      for (int e = 0; e < 16; ++e)
        o_tile[e] = TT::mfma16(__builtin_bit_cast(x8, op[e >> 1]), __builtin_bit_cast(x8, pB[e & 1]), o_tile[e]);
      // The copies of the steps past the row's end (the loop asks for K four and V two steps ahead,
      // whatever is left of the row) are still in flight: they must have landed before the epilogue
      // lays the finished row out in the same LDS.  (Nothing else waits for them: the barrier below
      // orders LDS accesses, not these copies, which the compiler does not see.)
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    } else {
    // Q operand.  A lane needs q row l32 of its sub-tile, 16 bytes out of every 32 (fp8: 32 of 64):
    // fetched straight from memory that is 64 scattered pieces per instruction (measured: ~4 k
    // cycles per row).  The 128 q rows are copied into LDS like a K tile instead (64 rows per kv
    // group, into the V half of its stage 1, which is free until the first MFMA block) and read
    // from there.  Requested first so that the latency overlaps the staging below.
    x8 qreg[kFp8 ? 1 : 8];
    i32x8 qreg8[kFp8 ? 2 : 1];
    i32x8 qlo8[kQLo ? 2 : 1];
    const uint32_t lds_group = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)group_smem));
    if constexpr (kFp8) {
      // (fp8 Q, half the bytes, is still fetched directly: with the LDS detour hipcc arranges the
      // main loop of this instantiation less well, which costs more than the detour saves)
      const uint8_t* src = qp + q_tok * p.q_sn + static_cast<int64_t>(my_head) * p.q_sh + g_p * 32;
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        const i32x4 lo = *reinterpret_cast<const i32x4*>(src + sl * 64);
        const i32x4 hi = *reinterpret_cast<const i32x4*>(src + sl * 64 + 16);
        qreg8[sl] = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
      if constexpr (kQLo) {
        const uint8_t* src2 = static_cast<const uint8_t*>(p.q_lo) + q_tok * p.q_sn +
                              static_cast<int64_t>(my_head) * p.q_sh + g_p * 32;
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
          const i32x4 lo = *reinterpret_cast<const i32x4*>(src2 + sl * 64);
          const i32x4 hi = *reinterpret_cast<const i32x4*>(src2 + sl * 64 + 16);
          qlo8[sl] = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
      }
    } else {
      const uint8_t* q_head = reinterpret_cast<const uint8_t*>(
          qp + static_cast<int64_t>(q_begin) * p.q_sn + static_cast<int64_t>(head_q0) * p.q_sh);
      const uint32_t qdst = lds_group + kStageBytes + kKBytes + qs * 1024;
      const int ln_q = fresh_lane();
      const int cp_row = ln_q >> 4, cp_chunk = ((ln_q & 15) ^ swz(4 * qs + cp_row)) * 8;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        int r = kg * 64 + 4 * (4 * n + qs) + cp_row;
        r = r < q_rows ? r : q_rows - 1;  // ragged last q block: re-read the last row
        copy16_to_lds(q_head, static_cast<uint32_t>((row_off(r, p.q_sn, p.q_sh) + cp_chunk) * sizeof(T)),
                      qdst + n * 4096);
      }
    }
    // (the row's kv block list is in LDS already: the main loop has no global loads besides the
    // tile copies, whose completion it tracks by counting, s_waitcnt vmcnt)
    // number of 64-key tiles; only the last listed block can be the request's ragged tail
    int n_tiles = 2 * nb;
    if (kv_len - s_blk[nb - 1] * kBlockKV <= kTileKV) n_tiles -= 1;
    const int my_tiles = (n_tiles - kg + 1) >> 1;  // tiles kg, kg+2, ...

    // softmax scale in the log2 domain; with fp8 operands the per-block dequantisation scales of
    // q (one per row of the list) and k (one per kv block) are folded in tile by tile
    float cq = c;
    if constexpr (kFp8) cq *= __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, ri.q_scale)));
    const int kv_head = head / p.kv_group;
    const float* const s_ksc = s_ksc2[row_it & 1];

    // Running reference point m_run of the softmax (log2 domain), partial sum d_part.  S^T is formed
    // relative to m_run: the MFMA accumulator starts at -m_run (c_init), so p = exp2(S^T) directly.
    // m_run is set to the tile's exact row max on the first tile and afterwards only raised when a
    // row's new max exceeds it by more than kLazyLog2 (p then stays <= 2^kLazyLog2, harmless in
    // fp32 / bf16 / fp16): the rescale of O leaves the steady-state path.
    f32x16 c_init;
#pragma unroll
    for (int i = 0; i < 16; ++i) c_init[i] = 0.f;

    // Tile copies.  The address of a copy is a wavefront-uniform tile base plus a per-lane byte
    // offset that does not change from tile to tile (row inside the tile, swizzled chunk); only a
    // request's ragged last tile clamps rows.  Tile j of this kv group = 64 keys of block j of the
    // row's list; it lives in LDS stage j & 1.  K and V of a tile are copied at different times,
    // each as early as its half of the stage is free:
    //   K of tile j+2 at the start of the VALU block of tile j   (K of tile j was consumed by S(j))
    //   V of tile j+1 during the MFMA block of tile j            (V of tile j-1 is in registers)
    // so a K copy has about two block periods to land and a V copy more than one.
    const TQK* k_head = kp + static_cast<int64_t>(kv_begin) * p.k_sn + static_cast<int64_t>(kv_head) * p.k_sh;
    const T* v_head = vp + static_cast<int64_t>(kv_begin) * p.v_sn + static_cast<int64_t>(kv_head) * p.v_sh;
    // lane offsets of copy instruction 0; instruction n adds a uniform 16 (fp8 K: 32) rows
    const uint32_t v_voff = static_cast<uint32_t>((4 * qs + cp_row) * p.v_sn + cp_chunk) * sizeof(T);
    const uint32_t k_voff = kFp8 ? static_cast<uint32_t>((8 * qs + cp8_row) * p.k_sn + cp8_chunk)
                                 : static_cast<uint32_t>((4 * qs + cp_row) * p.k_sn + cp_chunk) * sizeof(T);
    const int64_t k_jstep = (kFp8 ? 32 : 16) * p.k_sn * static_cast<int64_t>(sizeof(TQK));
    const int64_t v_jstep = 16 * p.v_sn * static_cast<int64_t>(sizeof(T));
    constexpr int kKCopies = (kFp8 && !kKLo) ? 2 : 4, kVCopies = 4;  // copy instructions per wavefront and tile
    const uint8_t* klo_head = nullptr;
    if constexpr (kKLo)
      klo_head = static_cast<const uint8_t*>(p.k_lo) + static_cast<int64_t>(kv_begin) * p.k_sn +
                 static_cast<int64_t>(kv_head) * p.k_sh;
    auto tile_start = [&](int j) { return s_blk[j] * kBlockKV + kg * kTileKV; };
    auto tile_valid = [&](int j) { return min(kTileKV, kv_len - tile_start(j)); };
    // all K copies of tile j at once
    auto copy_k = [&](int j) {
      const int start = __builtin_amdgcn_readfirstlane(tile_start(j));
      const int valid = min(kTileKV, kv_len - start);
      const uint8_t* kt = reinterpret_cast<const uint8_t*>(k_head + static_cast<int64_t>(start) * p.k_sn);
      const uint32_t kdst = lds_group + (j & 1) * kStageBytes + qs * 1024;
      // (two-term k: copy instructions 0, 1 fetch the tile of k, 2, 3 that of k_lo behind it)
      constexpr int kPerTerm = kKLo ? 2 : kKCopies;
      const uint8_t* kt_lo = kKLo ? klo_head + static_cast<int64_t>(start) * p.k_sn : nullptr;
      if (__builtin_expect(valid == kTileKV, 1)) {
#pragma unroll
        for (int n = 0; n < kKCopies; ++n)
          copy16_to_lds((n < kPerTerm ? kt : kt_lo) + (n % kPerTerm) * k_jstep, k_voff, kdst + n * 4096);
      } else {
        // ragged tail: re-read the last valid row, never overrun
        const int ln_c = fresh_lane();
        const int cp_row = ln_c >> 4, cp_chunk = ((ln_c & 15) ^ swz(4 * qs + cp_row)) * 8;
        const int cp8_row = ln_c >> 3, cp8_chunk = ((ln_c & 7) ^ ((4 * (qs & 1) + (ln_c >> 4)) & 7)) * 16;
#pragma unroll
        for (int n = 0; n < kKCopies; ++n) {
          int r = (kFp8 ? 8 : 4) * (4 * (n % kPerTerm) + qs) + (kFp8 ? cp8_row : cp_row);
          r = r < valid ? r : valid - 1;
          const uint32_t off = kFp8 ? static_cast<uint32_t>(r * p.k_sn + cp8_chunk)
                                    : static_cast<uint32_t>((r * p.k_sn + cp_chunk) * sizeof(T));
          copy16_to_lds(n < kPerTerm ? kt : kt_lo, off, kdst + n * 4096);
        }
      }
    };
    // V copies of tile j: prepared once, then issued one instruction at a time between MFMAs (a
    // wavefront that issues its share in one burst sits in the issue stage while the CU's address
    // unit, 64 B/clk, works through the burst of all eight wavefronts)
    const uint8_t* cp_v = nullptr;
    uint32_t cp_vdst = 0;
    bool cp_pending = false;
    int cp_valid = kTileKV;
    // scalar part (any time: it touches no LDS stage)
    auto copy_v_address = [&](int j) {
      const int start = __builtin_amdgcn_readfirstlane(tile_start(j));
      cp_valid = min(kTileKV, kv_len - start);
      cp_v = reinterpret_cast<const uint8_t*>(v_head + static_cast<int64_t>(start) * p.v_sn);
      cp_vdst = lds_group + (j & 1) * kStageBytes + kKBytes + qs * 1024;
    };
    // once the target stage is free: arm the one-by-one issue, or issue a ragged tile at once
    auto copy_v_prepare = [&]() {
      const int valid = cp_valid;
      cp_pending = valid == kTileKV;
      if (__builtin_expect(!cp_pending, 0)) {
        const int ln_c = fresh_lane();
        const int cp_row = ln_c >> 4, cp_chunk = ((ln_c & 15) ^ swz(4 * qs + cp_row)) * 8;
#pragma unroll
        for (int n = 0; n < kVCopies; ++n) {
          int r = 4 * (4 * n + qs) + cp_row;
          r = r < valid ? r : valid - 1;
          copy16_to_lds(cp_v, static_cast<uint32_t>((r * p.v_sn + cp_chunk) * sizeof(T)), cp_vdst + n * 4096);
        }
      }
    };
    auto copy_v_issue = [&](int n) {
      if (cp_pending) copy16_to_lds(cp_v + n * v_jstep, v_voff, cp_vdst + n * 4096);
    };
    // wait until at most n of this wavefront's copy instructions are outstanding (they complete in
    // issue order, so "the copies issued after X" outstanding means X has landed)
    auto wait_copies = [&](int n) {
      if (n >= 8) {
        __builtin_amdgcn_s_waitcnt(0x0f70 | 8);
      } else if (n >= 6) {
        __builtin_amdgcn_s_waitcnt(0x0f70 | 6);
      } else if (n >= 4) {
        __builtin_amdgcn_s_waitcnt(0x0f70 | 4);
      } else {
        __builtin_amdgcn_s_waitcnt(0x0f70);
      }
    };

    // ---- main loop: two-phase ("ping-pong") schedule ----
    // A wavefront alternates between an MFMA block (P.V of the previous tile, then K.Q^T of the
    // next) and a VALU block (online softmax).  The two kv groups share the SIMDs (wavefront w and
    // w+4 sit on SIMD w%4) and run half a period apart: every block starts at a workgroup barrier
    // and kv group 1 takes one extra barrier up front, so while one group's wavefronts feed the
    // matrix cores the other group's run their softmax on the vector ALUs.
    //   barrier calls: group 0 makes 2*T0 + 1, group 1 makes 1 + 2*T1 + 1 (T = tiles of the group);
    //   both pad to the larger count before the merge.
    const int calls_mine = kg == 0 ? 2 * ((n_tiles + 1) >> 1) + 1 : 2 * (n_tiles >> 1) + 2;
    const int calls_all = max(2 * ((n_tiles + 1) >> 1) + 1, 2 * (n_tiles >> 1) + 2);
    // copy order of a wavefront: K0, V0, K1 | V1 (MFMA block 0) | K2 (VALU block 0) | V2 | K3 | ...
    if (my_tiles > 0) {
      copy_k(0);
      copy_v_address(0);
      copy_v_prepare();
#pragma unroll
      for (int n = 0; n < kVCopies; ++n) copy_v_issue(n);
      cp_pending = false;
      if (my_tiles > 1) {
        copy_k(1);
        copy_v_address(1);
      }
    }
    // Q has landed once only the tile copies issued after it are outstanding; then for every
    // wavefront after the barrier
    if constexpr (!kFp8) {
      if (my_tiles > 1) {
        __builtin_amdgcn_s_waitcnt(0x0f70 | (2 * kKCopies + kVCopies));
      } else if (my_tiles == 1) {
        __builtin_amdgcn_s_waitcnt(0x0f70 | (kKCopies + kVCopies));
      } else {
        __builtin_amdgcn_s_waitcnt(0x0f70);
      }
    }
    __builtin_amdgcn_s_barrier();
    // Q from LDS while the first tile copies are in flight: rows (qs % 2) * 32 + l32 of the tile that
    // kv group qs / 2 copied, addressed like a K operand
    if constexpr (!kFp8) {
      // (the lane terms are made opaque here: otherwise the eight read addresses are worked out once
      // per kernel, live across the main loop, and their reloads wait for every copy in flight)
      const int ln_r = fresh_lane();
      const int q_rd_base = (ln_r & 31) * kRowBytes, q_rd_x = ((ln_r >> 5) ^ swz(ln_r & 31)) << 4;
      const uint8_t* qt = smem + (qs >> 1) * kGroupBytes + kStageBytes + kKBytes + (qs & 1) * 32 * kRowBytes +
                          q_rd_base;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) qreg[ks] = *reinterpret_cast<const x8*>(qt + (q_rd_x ^ (ks << 5)));
      // the softmax scale (log2 domain) is folded into Q, so S^T needs no multiply
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) qreg[ks][e] = static_cast<T>(static_cast<float>(qreg[ks][e]) * c);
    }
    // (every wavefront holds its Q before the first barrier: the V copies of tile 1 overwrite it after)
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    if (kg == 1) __builtin_amdgcn_s_barrier();

    f32x16 s[2];
    x8 vop[4][4], pb[4];

    // K operand reads of stage `it & 1`, d slices ks0..ks0+3 of both 32-key halves (16-bit K):
    // kop[h][ks - ks0] = rows h*32 + l32, d = ks*16 + g*8 .. +7
    auto read_k = [&](int it, int ks0, x8 (&kop)[2][4]) {
      const uint8_t* ks_base = group_smem + (it & 1) * kStageBytes + k_rd_base;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          kop[h][j] = *reinterpret_cast<const x8*>(ks_base + h * 32 * kRowBytes + (k_rd_x ^ ((ks0 + j) << 5)));
    };
    // four d slices of S^T for both 32-key halves; the two accumulator chains alternate so that no
    // MFMA waits for the one issued just before it
    auto s_math = [&](int ks0, const x8 (&kop)[2][4], int j0) {  // d slices ks0+j0, ks0+j0+1
#pragma unroll
      for (int j = j0; j < j0 + 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          s[h] = TT::mfma(kop[h][j], qreg[ks0 + j], (ks0 + j) == 0 ? c_init : s[h]);
    };
    // fp8: S^T straight from LDS (four reads, four MFMAs)
    auto s_fp8 = [&](int it) {
      if constexpr (kFp8) {
        const uint8_t* ks_base = group_smem + (it & 1) * kStageBytes;
        i32x8 k8[2][2];  // [32-key tile][64-wide d slab]: 32 consecutive fp8 of row l32
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int sl = 0; sl < 2; ++sl) {
            const uint8_t* rowp = ks_base + mt * 32 * kRowBytes8 + k_rd_base;
            const i32x4 lo = *reinterpret_cast<const i32x4*>(rowp + (k_rd_x ^ (sl << 6)));
            const i32x4 hi = *reinterpret_cast<const i32x4*>(rowp + ((k_rd_x ^ (sl << 6)) ^ 16));
            k8[mt][sl] = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
          for (int i = 0; i < 16; ++i) s[mt][i] = 0.f;
#pragma unroll
          for (int sl = 0; sl < 2; ++sl)
            s[mt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(k8[mt][sl], qreg8[sl], s[mt], 0, 0, 0,
                                                                    0x7f7f7f7f, 0, 0x7f7f7f7f);
        }
        if constexpr (kQLo) {
          // (second pass so that the two accumulator chains keep alternating)
#pragma unroll
          for (int sl = 0; sl < 2; ++sl)
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
              s[mt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(k8[mt][sl], qlo8[sl], s[mt], 0, 0, 0,
                                                                      0x7f7f7f7f, 0, 0x7f7f7f7f);
        }
        if constexpr (kKLo) {
          // k_lo . q^T: the tile of k_lo sits behind the tile of k in the stage
#pragma unroll
          for (int sl = 0; sl < 2; ++sl)
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
              const uint8_t* rowp = ks_base + kTileKV * kRowBytes8 + mt * 32 * kRowBytes8 + k_rd_base;
              const i32x4 lo = *reinterpret_cast<const i32x4*>(rowp + (k_rd_x ^ (sl << 6)));
              const i32x4 hi = *reinterpret_cast<const i32x4*>(rowp + ((k_rd_x ^ (sl << 6)) ^ 16));
              const i32x8 kl = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
              s[mt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(kl, qreg8[sl], s[mt], 0, 0, 0,
                                                                      0x7f7f7f7f, 0, 0x7f7f7f7f);
            }
        }
      }
    };
    // O^T += V^T . P^T for 16-key slabs kk0, kk0+1
    auto pv_math = [&](int kk) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o_acc[dt] = TT::mfma(vop[kk][dt], pb[kk], o_acc[dt]);
    };
    // VALU block of tile `it`: all V^T operands of the tile (4 slabs of 16 keys x 4 d tiles) are
    // requested first and land during the softmax
    auto valu_block = [&](int it, bool first) {
      // V of tile `it` has landed once only the copies issued after it (K and V of tile it+1) are
      // outstanding; after the barrier that holds for the whole kv group, and the group is done
      // reading K of this stage, which tile it+2 may now overwrite
      __builtin_amdgcn_s_setprio(0);
      wait_copies(it + 1 < my_tiles ? kKCopies + kVCopies : 0);
      __builtin_amdgcn_s_barrier();
      if (it + 2 < my_tiles) copy_k(it + 2);
      const int valid = tile_valid(it);
      float cs = cq;
      if constexpr (kFp8) cs = cq * s_ksc[it];
      const uint8_t* vs_base = group_smem + (it & 1) * kStageBytes + kKBytes;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const uint8_t* base = vs_base + kk * 16 * kRowBytes;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          union {
            s16x4 h[2];
            x8 v;
          } a;
          a.h[0] = lds_read_tr16(base + v_rd_off[dt][0]);
          a.h[1] = lds_read_tr16(base + v_rd_off[dt][1]);
          vop[kk][dt] = a.v;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      // online softmax (per lane: one q column, 32 kv values), log2 domain.  s holds x - m_run
      // (fp8: raw dot products, scaled and shifted here because the scale changes per kv block)
      if constexpr (kFp8) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[mt][i] = __builtin_fmaf(s[mt][i], cs, -m_run);
      }
      if constexpr (kCap) {
        // s holds 2 x log2(e) of tanh's argument x (the accumulators start at zero here):
        // tanh(x) = 1 - 2 / (1 + exp(2x)); score = cap_log2 * tanh(x), taken relative to m_run
        const float a = -2.f * p.cap_log2, b = p.cap_log2 - m_run;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[mt][i] = __builtin_fmaf(__builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[mt][i])), a, b);
      }
      if (valid < kTileKV) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int kv = mt * 32 + (i >> 2) * 8 + g * 4 + (i & 3);
            if (kv >= valid) s[mt][i] = -INFINITY;  // p = 0
          }
      }
      float mx = s[0][0];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[mt][i]);
      mx = max_across_halves(mx);  // row max relative to m_run
      if (first || __builtin_expect(__any(mx > kLazyLog2), 0)) {
        const float delta = first ? mx : fmaxf(mx, 0.f);
        if (!first) {
          const float scale = __builtin_amdgcn_exp2f(-delta);
          d_part *= scale;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o_acc[dt][i] *= scale;
        }
        m_run += delta;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[mt][i] -= delta;
        if constexpr (!kCap) {
#pragma unroll
          for (int i = 0; i < 16; ++i) c_init[i] = -m_run;
        }
      }
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          pb[mt * 2 + (i >> 3)][i & 7] = static_cast<T>(__builtin_amdgcn_exp2f(s[mt][i]));
      // the row sum is taken over the rounded p, as the reference does
      float psum = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) psum = TT::add_elems(pb[j], psum);
      d_part += psum;
      if (it + 2 < my_tiles) copy_v_address(it + 2);  // for the V copies of the next MFMA block
      __builtin_amdgcn_sched_barrier(0);
    };
    // start of an MFMA block: K of tile `it` has landed once only the copies issued after it (V of
    // this tile, K of the next) are outstanding, and this wavefront's V^T reads of the previous tile
    // have returned; after the barrier both hold for the whole kv group, so the V half of the other
    // stage may be overwritten
    auto open_mfma_block = [&](int it) {
      wait_copies(kVCopies + (it + 1 < my_tiles ? kKCopies : 0));
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_setprio(3);  // the MFMA block outranks the other kv group's softmax at issue
      cp_pending = false;
      if (it + 1 < my_tiles) copy_v_prepare();  // addresses were worked out in the last softmax block
    };
    // four MFMAs are followed by one copy instruction of the next tile
    auto after4 = [&](int n) {
      if (n < kVCopies) copy_v_issue(n);
      __builtin_amdgcn_sched_barrier(0);
    };

    if (my_tiles > 0) {
      // first tile: nothing to multiply by V yet
      open_mfma_block(0);
      if constexpr (kFp8) {
        s_fp8(0);
#pragma unroll
        for (int n = 0; n < 8; ++n) after4(n);
      } else {
        x8 k_lo[2][4], k_hi[2][4];
        read_k(0, 0, k_lo);
        read_k(0, 4, k_hi);
        __builtin_amdgcn_sched_barrier(0);
        s_math(0, k_lo, 0);
        after4(0);
        after4(1);
        s_math(0, k_lo, 2);
        after4(2);
        after4(3);
        s_math(4, k_hi, 0);
        after4(4);
        after4(5);
        s_math(4, k_hi, 2);
        after4(6);
        after4(7);
      }
      valu_block(0, true);
      for (int it = 1; it < my_tiles; ++it) {
        open_mfma_block(it);
        if constexpr (kFp8) {
          pv_math(0);
          after4(0);
          pv_math(1);
          after4(1);
          pv_math(2);
          after4(2);
          pv_math(3);
          after4(3);
          s_fp8(it);
        } else {
          // K operands are fetched under the MFMAs, half of them at a time, into the registers that
          // the V^T operands free
          x8 k_lo[2][4], k_hi[2][4];
          pv_math(0);
          after4(0);
          pv_math(1);
          after4(1);
          read_k(it, 0, k_lo);
          __builtin_amdgcn_sched_barrier(0);
          pv_math(2);
          after4(2);
          pv_math(3);
          after4(3);
          read_k(it, 4, k_hi);
          __builtin_amdgcn_sched_barrier(0);
          s_math(0, k_lo, 0);
          after4(4);
          s_math(0, k_lo, 2);
          after4(5);
          s_math(4, k_hi, 0);
          after4(6);
          s_math(4, k_hi, 2);
          after4(7);
        }
        valu_block(it, false);
      }
      // last MFMA block: P.V of the last tile
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_setprio(3);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) pv_math(kk);
      __builtin_amdgcn_s_setprio(0);
    } else {
      __builtin_amdgcn_s_barrier();
    }
    for (int i = calls_mine; i < calls_all; ++i) __builtin_amdgcn_s_barrier();
    if (my_tiles == 0) m_run = kNegInf;  // nothing seen: weight 0 in the merge
    }  // !kPipe

    // ---- merge the two kv groups through LDS, then write the row ----
    // (this lane's row, worked out again: what the prologue derived from the lane index would have
    // to live through the main loop, i.e. in scratch memory)
    const int lane_m = fresh_lane();
    const int l32_e = lane_m & 31, g_e = lane_m >> 5;
    const bool row_ok_e = qs * 32 + l32_e < q_rows;
    int tok_e, hq_e;
    row_at(row_ok_e ? qs * 32 + l32_e : q_rows - 1, tok_e, hq_e);
    const int64_t q_tok_e = q_begin + tok_e;
    const int my_head_e = head_q0 + hq_e;
    __syncthreads();  // all tile reads done: the tile buffers can be reused
    f32x4* mo = reinterpret_cast<f32x4*>(smem);
    float* md = reinterpret_cast<float*>(smem + kMergeOBytes);
    if constexpr (kGroups == 2) {
      if (kg == 1) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int i4 = 0; i4 < 4; ++i4) {
            f32x4 t4;
#pragma unroll
            for (int j = 0; j < 4; ++j) t4[j] = o_acc[dt][i4 * 4 + j];
            mo[(qs * 16 + dt * 4 + i4) * 64 + lane_m] = t4;
          }
        md[(qs * 64 + lane_m) * 2 + 0] = m_run;
        md[(qs * 64 + lane_m) * 2 + 1] = d_part;
      }
      __syncthreads();
    }
    if (wv == kFetchWave) {
      if constexpr (!kDirect) fetch_next((row_it + 1) & 1, false);
      else if constexpr (!kPipe) direct_next((row_it + 1) & 1);
    }
    // kv group 0: row maximum and row sum over both groups (kPipe: of the lane's two q rows)
    constexpr int kQ = kPipe ? 2 : 1;
    float m_all[kQ] = {}, d_all[kQ] = {};
    // the accumulators as 16 vectors of four d of one q row, vector e of q row e % kQ of the lane
    auto o_get = [&](int e, int j) __attribute__((always_inline)) {
      if constexpr (kPipe) return static_cast<float>(o_tile[e][j]);
      else return static_cast<float>(o_acc[e >> 2][(e & 3) * 4 + j]);
    };
    // (kPipe: lane l < 32 has the value of q row l)
    auto of_lane = [&](const float (&x)[kQ]) __attribute__((always_inline)) { 
      const float low = x[0], high = x[kQ - 1];
      return kPipe && (lane_m & 16) ? high : low;
    };
    // A lane owns one q row (kPipe: two) and runs of four d: stored from here, a row would leave as scattered
    // 8-byte pieces per instruction (measured: ~12 k cycles per row).  The finished row goes through
    // a padded LDS tile instead and leaves in 16-byte pieces, 16 consecutive lanes per 256-byte row.
    int ln_out = lane_m;
    asm volatile("" : "+v"(ln_out));  // (not hoisted out of the row loop and spilled)
    constexpr int kTileRows = kPipe ? 16 : 32;
    uint8_t* const out_row = smem + G::kOutOff + (qs * 32 + ln_out % kTileRows) * kOutRowBytes + ln_out / kTileRows * 8;
    auto out_at = [&](int e) __attribute__((always_inline)) {
      return reinterpret_cast<x4*>(kPipe ? out_row + (e & 1) * 16 * kOutRowBytes + (e >> 1) * 32 : out_row + e * 16);
    };
    bool store_row = parts == 1;
    if constexpr (kGroups == 1) {
      // one kv group: the accumulators hold the whole row
      float d_tot[kQ], inv[kQ];
#pragma unroll
      for (int i = 0; i < kQ; ++i) {
        const float d_half = d_q[i] + __shfl_xor(d_q[i], 16, 64);
        d_tot[i] = d_half + __shfl_xor(d_half, 32, 64);
        inv[i] = __builtin_amdgcn_rcpf(d_tot[i]);
        m_all[i] = m_q[i];
        d_all[i] = d_tot[i];
      }
      if (!kDirect || parts == 1) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          x4 out;
#pragma unroll
          for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(o_get(e, j) * inv[e % kQ]);
          *out_at(e) = out;
        }
        if (row_ok_e && p.lse && g_e == 0)
          p.lse[q_tok_e * p.num_heads + my_head_e] = __builtin_amdgcn_logf(of_lane(d_all)) + of_lane(m_all);
      }
    }
    if (kGroups == 2 && kg == 0) {
      const float m1 = md[(qs * 64 + lane_m) * 2 + 0], d1 = md[(qs * 64 + lane_m) * 2 + 1];
      const float m = fmaxf(m_run, m1);
      const float a0 = __builtin_amdgcn_exp2f(m_run - m);
      const float a1 = __builtin_amdgcn_exp2f(m1 - m);
      const float d_lane = d_part * a0 + d1 * a1;
      const float d_tot = d_lane + __shfl_xor(d_lane, 32, 64);
      if (parts == 1) {
        const float inv = __builtin_amdgcn_rcpf(d_tot);
        const float w0 = a0 * inv, w1 = a1 * inv;
        // all sixteen reads of the partner's partial first (the registers of the tile operands are
        // free here), so their latencies overlap
        f32x4 t4[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) t4[e] = mo[(qs * 16 + e) * 64 + lane_m];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          x4 out;
#pragma unroll
          for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(o_get(e, j) * w0 + t4[e][j] * w1);
          *out_at(e) = out;
        }
        if (row_ok_e && p.lse && g_e == 0)
          p.lse[q_tok_e * p.num_heads + my_head_e] = __builtin_amdgcn_logf(d_tot) + m;
      } else {
        // one part of a row cut at share boundaries: fold kv group 1 in without normalising; the
        // accumulators then hold this workgroup's partial result (reference point m, sum d_tot)
        f32x4 t4[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) t4[e] = mo[(qs * 16 + e) * 64 + lane_m];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            o_acc[e >> 2][(e & 3) * 4 + j] = o_acc[e >> 2][(e & 3) * 4 + j] * a0 + t4[e][j] * a1;
        m_all[0] = m;
        d_all[0] = d_tot;
      }
    }
    if ((kGroups == 2 || kDirect) && parts > 1) {
      // Whoever comes last combines the parts and writes the row.  A workgroup that finds every
      // other part arrived already need not publish its own; otherwise it publishes, then counts
      // itself in, and may still turn out to be the last.
      // (Even shares: the first item of a share is the end of a row that began in another share, whose last item its beginning
      // is.  It is early, and does not ask.)
      bool last = false;
      if (!kDirect || row_it > 0 || part == 0) {
        if (tid == 0)
          s_arrived = __hip_atomic_load(&p.sched[kSchedArrived + split_slot], __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        last = s_arrived == parts - 1;
      }
      if (!last) {
        if (kg == 0) {
          // same lane layout as the LDS merge area; two planes of 8-byte pairs, so that each store
          // instruction covers 512 contiguous bytes
          float* part_ws = p.split_ws + static_cast<int64_t>(part_area(split_slot, part)) * kSplitPartFloats;
          const int ln = fresh_lane();
          float* lane_ws = part_ws + (qs * 16 * 2 * 64 + ln) * 2;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            store_pair_device(lane_ws + e * 256, o_get(e, 0), o_get(e, 1));
            store_pair_device(lane_ws + e * 256 + 128, o_get(e, 2), o_get(e, 3));
          }
          store_pair_device(part_ws + 128 * 128 + (qs * 64 + ln) * 2, of_lane(m_all), of_lane(d_all));
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this lane's partial results have left
        __syncthreads();
        if (tid == 0) s_arrived = atomicAdd(&p.sched[kSchedArrived + split_slot], 1);
        __syncthreads();
        last = s_arrived == parts - 1;
      }
      if (last) {
        if (kg == 0) {
          // The parts are added in part order, this workgroup's own from its registers (the same
          // values it would have published), the others read back: the row does not depend on
          // which part came last.
          auto part_base = [&](int i) {
            return p.split_ws + static_cast<int64_t>(part_area(split_slot, i)) * kSplitPartFloats;
          };
          // (a part's maximum and sum are read twice: held in an array, they would be in scratch memory)
          float m_own[kQ], d_own[kQ];
#pragma unroll
          for (int q = 0; q < kQ; ++q) {
            m_own[q] = m_all[q];
            d_own[q] = d_all[q];
            m_all[q] = kNegInf;
            d_all[q] = 0.f;
          }
          auto part_stats = [&](int i, float (&m)[kQ], float (&d)[kQ]) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < kQ; ++q) {
              m[q] = m_own[q];
              d[q] = d_own[q];
              if (i != part)
                load_pair_device(part_base(i) + 128 * 128 + (qs * 64 + (kPipe ? 16 * q + (lane_m & 15) : lane_m)) * 2, m[q], d[q]);
            }
          };
          for (int i = 0; i < parts; ++i) {
            float m[kQ], d[kQ];
            part_stats(i, m, d);
#pragma unroll
            for (int q = 0; q < kQ; ++q) m_all[q] = fmaxf(m_all[q], m[q]);
          }
          f32x4 acc[16];
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
          const int ln = fresh_lane();
          for (int i = 0; i < parts; ++i) {
            float m[kQ], d[kQ], a[kQ];
            part_stats(i, m, d);
            if (i == part) {
#pragma unroll
              for (int q = 0; q < kQ; ++q) {
                a[q] = __builtin_amdgcn_exp2f(m[q] - m_all[q]);
                d_all[q] = __builtin_fmaf(d[q], a[q], d_all[q]);
              }
#pragma unroll
              for (int e = 0; e < 16; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[e][j] = __builtin_fmaf(o_get(e, j), a[e % kQ], acc[e][j]);
            } else {
              const float* lane_ws = part_base(i) + (qs * 16 * 2 * 64 + ln) * 2;
              // all loads of the part in flight together
              float u[16][4];
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                load_pair_device(lane_ws + e * 256, u[e][0], u[e][1]);
                load_pair_device(lane_ws + e * 256 + 128, u[e][2], u[e][3]);
              }
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int q = 0; q < kQ; ++q) {
                a[q] = __builtin_amdgcn_exp2f(m[q] - m_all[q]);
                d_all[q] = __builtin_fmaf(d[q], a[q], d_all[q]);
              }
#pragma unroll
              for (int e = 0; e < 16; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[e][j] = __builtin_fmaf(u[e][j], a[e % kQ], acc[e][j]);
            }
          }
          float inv[kQ];
#pragma unroll
          for (int q = 0; q < kQ; ++q) inv[q] = __builtin_amdgcn_rcpf(d_all[q]);
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            x4 out;
#pragma unroll
            for (int j = 0; j < 4; ++j) out[j] = static_cast<T>(acc[e][j] * inv[e % kQ]);
            *out_at(e) = out;
          }
          if (row_ok_e && p.lse && g_e == 0)
            p.lse[q_tok_e * p.num_heads + my_head_e] = __builtin_amdgcn_logf(of_lane(d_all)) + of_lane(m_all);
        }
        if (tid == 0) p.sched[kSchedArrived + split_slot] = 0;  // re-armed for the next launch
        store_row = true;
      }
      // (nothing may be in flight into registers where this path joins the one that stores a row:
      // the compiler would wait there for everything, the row's stores included)
      __builtin_amdgcn_s_waitcnt(0x0f70);
    }
    if (store_row && kg == 0) {
      // A wavefront stores the 32 rows it has just written to the LDS tile itself: no barrier, so
      // the other kv group (whose first wavefront is fetching the next row's record meanwhile) is not
      // waited for here but at the top of the next row.
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's rows are in the tile
      T* dst = op + static_cast<int64_t>(q_begin) * p.o_sn + static_cast<int64_t>(head_q0) * p.o_sh;
      // (the lane index is worked out afresh here: otherwise the per-lane address terms are computed once
      // per kernel, spilled, and every reload waits for the store before it)
      const int ln = fresh_lane();
      const int r0 = qs * 32 + (ln >> 4), chunk = ln & 15;
      u32x4 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[i] = *reinterpret_cast<const u32x4*>(smem + G::kOutOff + (r0 + i * 4) * kOutRowBytes + chunk * 16);
      T* d0 = dst + chunk * 8;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        // (streaming stores: O is not read again here and should not push K and V out of the L2;
        // 3 MB less fetched per FLUX-sized launch at the same speed.  The same hint on the Q copies
        // takes another 6 MB off and 0.6 % of speed: not used.)
        if (r0 + i * 4 < q_rows) __builtin_nontemporal_store(v[i], reinterpret_cast<u32x4*>(d0 + row_off(r0 + i * 4, p.o_sn, p.o_sh)));
    }
  }

  if constexpr (kDirect) {
    // q blocks that are not computed, of a fresh output: zeros (left to the end: a workgroup that has no row
    // comes here at once)
    const int n_zero = __builtin_amdgcn_readfirstlane(s_dir[1]);
    for (int z = 0; z < n_zero; ++z) {
      RowInfo it;
      direct_row(s_zero[z], it);
      const int gq = kGqaPack ? p.gqa_pack : 0;
      T* dst = op + static_cast<int64_t>(it.q_begin) * p.o_sn + static_cast<int64_t>(gq ? it.head * gq : it.head) * p.o_sh;
      for (int i = tid; i < it.q_rows * 16; i += 64 * kWaves) {
        const int r = i >> 4;
        int64_t off;
        if constexpr (kGqaPack) {
          const uint32_t pr = static_cast<uint32_t>(it.qb) * kBlockQ + r;
          const int tok = static_cast<int>(pr / static_cast<uint32_t>(gq));
          off = tok * p.o_sn + static_cast<int64_t>(pr - tok * gq) * p.o_sh;
        } else {
          off = r * p.o_sn;
        }
        const u32x4 zero = {0u, 0u, 0u, 0u};
        __builtin_nontemporal_store(zero, reinterpret_cast<u32x4*>(dst + off) + (i & 15));
      }
    }
    return;
  }
  // the last workgroup to leave rewinds the queues for the next launch
  // (every pop's answer has come back by now, so no fence is needed between the atomics; one writes the XCD's L2
  // back, once per workgroup)
  if (tid == 0) {
    const int done = atomicAdd(&p.sched[24], 1);
    if (done == static_cast<int>(gridDim.x) - 1) {
      for (int x = 0; x < kXcds; ++x) p.sched[16 + x] = 0;
      p.sched[24] = 0;
    }
  }
}

// The two-term fp8 k of a long list, widened once per call: k16 = k + k_lo in fp16, kv head by kv head
// ([num_kv_heads][n_kv_blocks][128][128], blocks numbered as in k_scale, so that the room does not depend on where the
// batch's tokens begin; a request's last block is filled as far as the request goes).  The fp8 form multiplies three
// times (k.q, k.q_lo, k_lo.q) in the two-phase loop; fp16 operands take one product in the pipelined loop.  All scales
// stay out of the operands: they are multiplied into S in fp32, block by block, as the fp8 form does.
// Precision: where a residual's bits lie within 11 of its value's first one the widened operand is the exact sum (it
// always is for values that e4m3 holds by themselves); a smaller residual (|lo| < 2^-7 of the binade: one value in
// eight) is rounded with an error of at most 2^-11 of the value, and the pair's own distance from the number it stands
// for is up to four times as much.  The fp8 form keeps every residual, and leaves k_lo.q_lo out of every logit.  Logits
// of 128 products against 64 bits, rms over the sum of the products' sizes, fp8 form and this: 9.4e-5 and 1.5e-5
// (normal data, whatever the blocks' scales), 4.4e-5 and 2.8e-8 (both on the e4m3 grid, a 448 among small values),
// 4.3e-6 and 1.2e-5 (q_lo all zero and k normal: here the fp8 form leaves nothing out; to the numbers that the pairs
// stand for both are equally far).
// What is left to the fp8 form, row by row: k scales of a head that are not positive and finite, and products of the
// scales outside of 2^-100 .. 2^90.
// 2 bytes read and 2 written per element: 0.3 ms for 76112 tokens x 40 heads, where the layer's call went from 17.3 to
// 14.8 ms.  (With the scales rounded into the operands, and the accumulators of S beginning at the softmax's reference
// point, 14.7.)
__global__ void __launch_bounds__(256) widen_k_kernel(
    const uint8_t* __restrict__ k, const uint8_t* __restrict__ k_lo, int64_t k_sn, int64_t k_sh,
    const float* __restrict__ k_scale, const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_blk_base,
    int32_t batch, int32_t n_kv_blocks, _Float16* __restrict__ k16, f32x2* __restrict__ range, int32_t* __restrict__ left) {
  __shared__ float s_max[4], s_min[4];
  __shared__ int s_req;
  const int blk = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid == 0) s_req = -1;
  __syncthreads();
  // the request of this block
  for (int r = tid; r < batch; r += 256)
    if (kv_blk_base[r] <= blk && blk < kv_blk_base[r + 1]) s_req = r;
  // a head's smallest and largest scale, by its first workgroup (one that is not positive and finite counts as infinite)
  if (blk == 0) {
    float mx = 0.f, mn = __builtin_inff();
    for (int i = tid; i < n_kv_blocks; i += 256) {
      const float v = k_scale[static_cast<int64_t>(head) * n_kv_blocks + i];
      mx = fmaxf(mx, v > 0.f ? v : __builtin_inff());
      mn = fminf(mn, v);
    }
    for (int off = 32; off > 0; off >>= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, off, 64));
      mn = fminf(mn, __shfl_xor(mn, off, 64));
    }
    if (lane == 0) {
      s_max[wv] = mx;
      s_min[wv] = mn;
    }
  }
  __syncthreads();
  if (blk == 0 && tid == 0) {
    range[head] = f32x2{fminf(fminf(s_min[0], s_min[1]), fminf(s_min[2], s_min[3])),
                        fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]))};
    if (head == 0) *left = 0;
  }
  const int req = s_req;
  if (req < 0) return;
  const int tok0 = kv_indptr[req] + (blk - kv_blk_base[req]) * kBlockKV;
  const int len = min(kBlockKV, kv_indptr[req + 1] - tok0);
  const int col = (tid & 7) * 16;
  _Float16* out = k16 + (static_cast<int64_t>(head) * n_kv_blocks + blk) * (kBlockKV * kHeadDim) + col;
  const int64_t in = static_cast<int64_t>(tok0) * k_sn + static_cast<int64_t>(head) * k_sh + col;
  u32x4 hi[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = min((tid >> 3) + 32 * i, len - 1);
    hi[i] = *reinterpret_cast<const u32x4*>(k + in + r * k_sn);
    lo[i] = *reinterpret_cast<const u32x4*>(k_lo + in + r * k_sn);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = (tid >> 3) + 32 * i;
    if (r < len) {
      f16x8 a, b;
      widen8(u32x2{hi[i][0], hi[i][1]}, u32x2{lo[i][0], lo[i][1]}, a);
      widen8(u32x2{hi[i][2], hi[i][3]}, u32x2{lo[i][2], lo[i][3]}, b);
      f16x8* dst = reinterpret_cast<f16x8*>(out + r * kHeadDim);
      dst[0] = a;
      dst[1] = b;
    }
  }
}

template <typename T, bool kFp8, bool kQLo, bool kKLo, int kGroups = 2, bool kPipe = false, bool kGqaPack = false,
          bool kCap = false, bool kDirect = false, bool kWide = false, int kMany = 0>
int launch(const FaParams& p, int64_t max_rows, hipStream_t stream) {
  constexpr int kSmemBytes = Geom<kFp8, kKLo, kGroups>::kSmemBytes;
  // (the attribute belongs to the kernel's code object on one device: set once per device; the flags
  // are atomic because host threads may launch concurrently, and setting it twice is harmless)
  static std::atomic<bool> attr_set[64] = {};
  int dev = 0;
  FO_HIP_CALL(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    FO_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(&sparse_fa_kernel<T, kFp8, kQLo, kKLo, kGroups, kPipe, kGqaPack, kCap, kDirect, kWide, kMany>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kSmemBytes));
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  int num_cu = fo_num_cu();
  if (num_cu <= 0) return fo::fail(FO_ERR_HIP, "sparse_fa: no device");
  int64_t grid = num_cu * (3 - kGroups);  // persistent workgroups: one per CU, or two of one kv group each (LDS bound)
  // (with even shares every workgroup may hold a part of a row; otherwise at most one row each)
  if (!kDirect && !(p.split_ws && p.shares) && grid > max_rows) grid = max_rows;
  sparse_fa_kernel<T, kFp8, kQLo, kKLo, kGroups, kPipe, kGqaPack, kCap, kDirect, kWide, kMany><<<static_cast<unsigned>(grid), kGroups * kGroupThreads, kSmemBytes, stream>>>(p);
  FO_CHECK_LAUNCH();
  return FO_OK;
}

}  // namespace

namespace {
std::atomic<int> g_variant{0};
}

extern "C" int fo_sparse_fa_set_variant(int variant) {
  FO_REQUIRE(variant >= 0 && variant <= 2, "sparse_fa: variant must be 0 (automatic), 1 or 2");
  g_variant.store(variant, std::memory_order_relaxed);
  return FO_OK;
}

extern "C" int64_t fo_sparse_fa_wide_bytes(int64_t max_rows, int32_t num_kv_heads, int32_t n_kv_blocks);

extern "C" int64_t fo_sparse_fa_split_workspace_bytes(void) {
  // two areas per share, one share per workgroup = per CU
  return static_cast<int64_t>(2) * fo_num_cu() * kSplitPartFloats * sizeof(float);
}

namespace {
// widened fp8 operands: the head of the workspace (the kv heads' ranges of scales and a word), then k16
int64_t wide_head_bytes(int32_t num_kv_heads) { return (static_cast<int64_t>(num_kv_heads) * 8 + 4 + 255) / 256 * 256; }
// the pipelined form is taken from this many rows on
bool long_list(int64_t max_rows) { return max_rows >= static_cast<int64_t>(8) * fo_num_cu(); }
bool wide_serves(int64_t max_rows, int32_t num_kv_heads, int32_t n_kv_blocks) {
  const int variant = g_variant.load(std::memory_order_relaxed);
  return (variant == 1 || (variant == 0 && long_list(max_rows))) && max_rows > 0 && num_kv_heads > 0 && num_kv_heads <= 65535 &&
         n_kv_blocks > 0 && n_kv_blocks <= kMaxRowBlocksOneGroup;
}

int run_decoded(const void* q, const void* k, const void* v, void* o, float* lse,
                                int dtype, const void* q_lo, const void* k_lo, const float* q_scale,
                                const float* k_scale,
                                int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                                int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                                int64_t o_stride_n, int64_t o_stride_h, const int32_t* qo_indptr,
                                const int32_t* kv_indptr, const int32_t* q_blk_base,
                                const int32_t* kv_blk_base, int32_t n_q_blocks,
                                int32_t n_kv_blocks, const int32_t* row_req,
                                const int32_t* row_qb, const int32_t* row_head,
                                const int32_t* kv_row_ptr, const int32_t* kv_idx,
                                const int32_t* order, int32_t* sched, int64_t max_rows,
                                int32_t num_heads, int32_t num_kv_heads, int32_t gqa_packed, int32_t head_dim,
                                int32_t block_q, int32_t block_kv, float sm_scale, float logits_soft_cap,
                                const int32_t* shares, void* split_workspace, int64_t split_workspace_bytes,
                                void* wide, int64_t wide_bytes, int32_t batch, void* stream) {
  FO_REQUIRE(head_dim == kHeadDim, "sparse_fa: head_dim %d is not supported (only 128)", head_dim);
  FO_REQUIRE(block_q == kBlockQ && block_kv == kBlockKV,
             "sparse_fa: sparse block sizes (%d, %d) are not supported (only 128, 128)", block_q,
             block_kv);
  FO_REQUIRE(dtype == FO_BF16 || dtype == FO_F16 || dtype == FO_FP8_E4M3,
             "sparse_fa: unsupported dtype code %d", dtype);
  FO_REQUIRE(num_heads > 0 && max_rows >= 0, "sparse_fa: bad sizes");
  FO_REQUIRE(num_kv_heads > 0 && num_heads % num_kv_heads == 0,
             "sparse_fa: num_qo_heads %d is not a multiple of num_kv_heads %d", num_heads, num_kv_heads);
  FO_REQUIRE(gqa_packed == 0 || gqa_packed == 1, "sparse_fa: gqa_packed must be 0 or 1");
  FO_REQUIRE(logits_soft_cap >= 0.f && logits_soft_cap < __builtin_inff(),
             "sparse_fa: logits_soft_cap must be a finite value >= 0 (0: no cap)");
  FO_REQUIRE(logits_soft_cap == 0.f || dtype != FO_FP8_E4M3, "sparse_fa: the logits soft cap is not built for fp8 q/k");
  FO_REQUIRE(!gqa_packed || dtype != FO_FP8_E4M3,
             "sparse_fa: fp8 q (one scale per q head and token block) is not built for packed tiles of "
             "several q heads");
  if (max_rows == 0) return FO_OK;
  FO_REQUIRE(q && k && v && o && qo_indptr && kv_indptr && row_req && row_qb && row_head &&
                 kv_row_ptr && kv_idx && order && sched,
             "sparse_fa: null pointer");
  const int64_t strides[8] = {q_stride_n, q_stride_h, k_stride_n, k_stride_h,
                              v_stride_n, v_stride_h, o_stride_n, o_stride_h};
  for (int i = 0; i < 8; ++i)
    FO_REQUIRE(strides[i] % (dtype == FO_FP8_E4M3 && i < 4 ? 16 : 8) == 0 && strides[i] > 0,
               "sparse_fa: strides must be positive multiples of 16 bytes (128-bit accesses)");
  FO_REQUIRE(q_stride_n < (int64_t(1) << 23) && k_stride_n < (int64_t(1) << 23) &&
                 v_stride_n < (int64_t(1) << 23),
             "sparse_fa: q/k/v token strides must be below 2^23 elements (32-bit tile offsets)");
  if (dtype == FO_FP8_E4M3)
    FO_REQUIRE(q_scale && k_scale && q_blk_base && kv_blk_base && n_q_blocks > 0 && n_kv_blocks > 0,
               "sparse_fa: fp8 q/k need q_scale, k_scale, the block numbering and the scale row lengths");
  FO_REQUIRE(q_lo == nullptr || dtype == FO_FP8_E4M3, "sparse_fa: q_lo is the second term of an fp8 q");
  FO_REQUIRE(k_lo == nullptr || q_lo != nullptr, "sparse_fa: k_lo (second term of an fp8 k) needs q_lo as well");
  for (const void* ptr : {q, k, v, static_cast<const void*>(o), q_lo, k_lo})
    FO_REQUIRE((reinterpret_cast<uintptr_t>(ptr) & 15) == 0,
               "sparse_fa: q/k/v/o must be 16-byte aligned");

  FaParams p{};
  p.q = q; p.k = k; p.v = v; p.o = o; p.lse = lse;
  p.q_lo = q_lo; p.k_lo = k_lo; p.q_scale = q_scale; p.k_scale = k_scale;
  p.q_sn = q_stride_n; p.q_sh = q_stride_h; p.k_sn = k_stride_n; p.k_sh = k_stride_h;
  p.v_sn = v_stride_n; p.v_sh = v_stride_h; p.o_sn = o_stride_n; p.o_sh = o_stride_h;
  p.qo_indptr = qo_indptr; p.kv_indptr = kv_indptr;
  p.q_blk_base = q_blk_base; p.kv_blk_base = kv_blk_base;
  p.row_req = row_req; p.row_qb = row_qb; p.row_head = row_head;
  p.kv_row_ptr = kv_row_ptr; p.kv_idx = kv_idx; p.order = order; p.sched = sched;
  // even shares need both the decoder's share table and room for partial results (without them
  // the rows are taken whole from the queues, which the decoder fills either way)
  p.split_ws = nullptr;
  p.shares = nullptr;
  if (shares != nullptr) {
    FO_REQUIRE(split_workspace != nullptr && split_workspace_bytes >= fo_sparse_fa_split_workspace_bytes(),
               "sparse_fa: the work list was decoded for even shares, which need a split workspace of "
               "fo_sparse_fa_split_workspace_bytes() bytes");
    FO_REQUIRE((reinterpret_cast<uintptr_t>(split_workspace) & 15) == 0,
               "sparse_fa: split_workspace must be 16-byte aligned");
    p.split_ws = static_cast<float*>(split_workspace);
    p.shares = shares;
  }
  p.num_heads = num_heads;
  // packed tiles: row_head is the kv head already, and a tile's rows spread over its q heads
  const bool packed = gqa_packed && num_heads != num_kv_heads;
  p.kv_group = packed ? 1 : num_heads / num_kv_heads;
  p.gqa_pack = packed ? num_heads / num_kv_heads : 0; p.n_q_blocks = n_q_blocks; p.n_kv_blocks = n_kv_blocks;
  p.sm_scale_log2 = sm_scale * 1.44269504088896340736f;
  p.cap_log2 = 0.f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (logits_soft_cap > 0.f) {
    // (reference: soft_cap_pre_tanh_scale = sm_scale / cap, sm_scale_log2 = log2(e) * cap, variants.cuh:43-56)
    p.cap_log2 = logits_soft_cap * 1.44269504088896340736f;
    p.sm_scale_log2 = 2.f * 1.44269504088896340736f * sm_scale / logits_soft_cap;
    if (p.gqa_pack)
      return dtype == FO_BF16 ? launch<__bf16, false, false, false, 2, false, true, true>(p, max_rows, s)
                              : launch<_Float16, false, false, false, 2, false, true, true>(p, max_rows, s);
    return dtype == FO_BF16 ? launch<__bf16, false, false, false, 2, false, false, true>(p, max_rows, s)
                            : launch<_Float16, false, false, false, 2, false, false, true>(p, max_rows, s);
  }
  // Long lists (many rows per CU) run as two independent 4-wavefront workgroups per CU with the
  // software-pipelined loop; short ones as one 8-wavefront workgroup whose two kv groups share a row
  // (half the latency per row, and rows can be cut into even shares).  The list's length lives on the
  // device: the choice is made from its upper bound max_rows, unless fo_sparse_fa_set_variant() fixed
  // it.  The one-group form needs 16-bit operands, at most 3072 kv blocks per request and kv spans
  // below 4 GiB (32-bit copy offsets): n_kv_blocks, the batch's total, bounds both.
  const int64_t span = static_cast<int64_t>(n_kv_blocks) * kBlockKV * 2;
  const bool one_group_ok = (dtype == FO_BF16 || dtype == FO_F16) && n_kv_blocks > 0 &&
                            n_kv_blocks <= kMaxRowBlocksOneGroup && span * k_stride_n < (int64_t(1) << 32) &&
                            span * v_stride_n < (int64_t(1) << 32);
  const int variant = g_variant.load(std::memory_order_relaxed);
  const bool one_group = one_group_ok && (variant == 1 || (variant == 0 && long_list(max_rows)));
  if (p.gqa_pack) {  // packed tiles of several q heads: the row mapping is compiled in
    if (dtype == FO_BF16)
      return one_group ? launch<__bf16, false, false, false, 1, true, true>(p, max_rows, s)
                       : launch<__bf16, false, false, false, 2, false, true>(p, max_rows, s);
    return one_group ? launch<_Float16, false, false, false, 1, true, true>(p, max_rows, s)
                     : launch<_Float16, false, false, false, 2, false, true>(p, max_rows, s);
  }
  if (dtype == FO_BF16)
    return one_group ? launch<__bf16, false, false, false, 1, true>(p, max_rows, s)
                     : launch<__bf16, false, false, false, 2>(p, max_rows, s);
  if (dtype == FO_F16)
    return one_group ? launch<_Float16, false, false, false, 1, true>(p, max_rows, s)
                     : launch<_Float16, false, false, false, 2>(p, max_rows, s);
  if (k_lo != nullptr) {
    if (wide != nullptr && wide_serves(max_rows, num_kv_heads, n_kv_blocks) && span * v_stride_n < (int64_t(1) << 32)) {
      FO_REQUIRE(batch > 0 && wide_bytes >= fo_sparse_fa_wide_bytes(max_rows, num_kv_heads, n_kv_blocks) &&
                     (reinterpret_cast<uintptr_t>(wide) & 255) == 0,
                 "sparse_fa: the workspace for widened operands must be 256-byte aligned and hold "
                 "fo_sparse_fa_wide_bytes() bytes");
      f32x2* range = static_cast<f32x2*>(wide);
      int32_t* left = reinterpret_cast<int32_t*>(range + num_kv_heads);
      _Float16* k16 = reinterpret_cast<_Float16*>(static_cast<uint8_t*>(wide) + wide_head_bytes(num_kv_heads));
      widen_k_kernel<<<dim3(n_kv_blocks, num_kv_heads), 256, 0, s>>>(
          static_cast<const uint8_t*>(k), static_cast<const uint8_t*>(k_lo), k_stride_n, k_stride_h, k_scale, kv_indptr,
          kv_blk_base, batch, n_kv_blocks, k16, range, left);
      FO_CHECK_LAUNCH();
      p.wide_range = range;
      p.wide_left = left;
      FaParams w = p;
      w.k = k16;
      w.k_sn = kHeadDim;
      const int rc = launch<__bf16, false, false, false, 1, true, false, false, false, true>(w, max_rows, s);
      if (rc != FO_OK) return rc;
    }
    return launch<__bf16, true, true, true>(p, max_rows, s);
  }
  if (q_lo != nullptr) return launch<__bf16, true, true, false>(p, max_rows, s);
  return launch<__bf16, true, false, false>(p, max_rows, s);
}

}  // namespace

extern "C" int fo_sparse_fa_run(const void* q, const void* k, const void* v, void* o, float* lse,
                                int dtype, const void* q_lo, const void* k_lo, const float* q_scale,
                                const float* k_scale,
                                int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                                int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                                int64_t o_stride_n, int64_t o_stride_h, const int32_t* qo_indptr,
                                const int32_t* kv_indptr, const int32_t* q_blk_base,
                                const int32_t* kv_blk_base, int32_t n_q_blocks,
                                int32_t n_kv_blocks, const int32_t* row_req,
                                const int32_t* row_qb, const int32_t* row_head,
                                const int32_t* kv_row_ptr, const int32_t* kv_idx,
                                const int32_t* order, int32_t* sched, int64_t max_rows,
                                int32_t num_heads, int32_t num_kv_heads, int32_t gqa_packed, int32_t head_dim,
                                int32_t block_q, int32_t block_kv, float sm_scale, float logits_soft_cap,
                                const int32_t* shares, void* split_workspace, int64_t split_workspace_bytes,
                                void* stream) {
  return run_decoded(q, k, v, o, lse, dtype, q_lo, k_lo, q_scale, k_scale, q_stride_n, q_stride_h, k_stride_n, k_stride_h,
                     v_stride_n, v_stride_h, o_stride_n, o_stride_h, qo_indptr, kv_indptr, q_blk_base, kv_blk_base, n_q_blocks,
                     n_kv_blocks, row_req, row_qb, row_head, kv_row_ptr, kv_idx, order, sched, max_rows, num_heads,
                     num_kv_heads, gqa_packed, head_dim, block_q, block_kv, sm_scale, logits_soft_cap, shares,
                     split_workspace, split_workspace_bytes, nullptr, 0, 0, stream);
}

extern "C" int fo_sparse_fa_run_wide(const void* q, const void* k, const void* v, void* o, float* lse,
                                int dtype, const void* q_lo, const void* k_lo, const float* q_scale,
                                const float* k_scale,
                                int64_t q_stride_n, int64_t q_stride_h, int64_t k_stride_n,
                                int64_t k_stride_h, int64_t v_stride_n, int64_t v_stride_h,
                                int64_t o_stride_n, int64_t o_stride_h, const int32_t* qo_indptr,
                                const int32_t* kv_indptr, const int32_t* q_blk_base,
                                const int32_t* kv_blk_base, int32_t n_q_blocks,
                                int32_t n_kv_blocks, const int32_t* row_req,
                                const int32_t* row_qb, const int32_t* row_head,
                                const int32_t* kv_row_ptr, const int32_t* kv_idx,
                                const int32_t* order, int32_t* sched, int64_t max_rows,
                                int32_t num_heads, int32_t num_kv_heads, int32_t gqa_packed, int32_t head_dim,
                                int32_t block_q, int32_t block_kv, float sm_scale, float logits_soft_cap,
                                const int32_t* shares, void* split_workspace, int64_t split_workspace_bytes,
                                void* wide, int64_t wide_bytes, int32_t batch, void* stream) {
  return run_decoded(q, k, v, o, lse, dtype, q_lo, k_lo, q_scale, k_scale, q_stride_n, q_stride_h, k_stride_n, k_stride_h,
                     v_stride_n, v_stride_h, o_stride_n, o_stride_h, qo_indptr, kv_indptr, q_blk_base, kv_blk_base, n_q_blocks,
                     n_kv_blocks, row_req, row_qb, row_head, kv_row_ptr, kv_idx, order, sched, max_rows, num_heads,
                     num_kv_heads, gqa_packed, head_dim, block_q, block_kv, sm_scale, logits_soft_cap, shares,
                     split_workspace, split_workspace_bytes, wide, wide_bytes, batch, stream);
}

extern "C" int64_t fo_sparse_fa_wide_bytes(int64_t max_rows, int32_t num_kv_heads, int32_t n_kv_blocks) {
  if (!wide_serves(max_rows, num_kv_heads, n_kv_blocks)) return 0;
  return wide_head_bytes(num_kv_heads) + static_cast<int64_t>(num_kv_heads) * n_kv_blocks * kBlockKV * kHeadDim * 2;
}

namespace {

int64_t direct_candidates(const fo_attention_args& a) { return static_cast<int64_t>(a.n_blk) * a.symbol_heads; }

// Two workgroups of four wavefronts per CU and the software-pipelined loop, whose row boundaries pass beside the other
// workgroup's main loop; where there are too few rows for that, the two-phase loop with twice the wavefronts per row.
// Two-phase against pipelined, us per call.  Where every row is computed (is_full) from 13/8 of a candidate per CU on:
//   416 candidates of 13 blocks 61.2 / 51.0    408 of 102 370 / 298    408 of 17 74.9 / 67.3    432 of 36 148 / 131
//   384 of 24 85.5 / 86.5    384 of 32 109 / 101    384 of 16 62.8 / 61.0
// With symbols the host does not know how many rows there are, and from 2.5 per CU on (with active rows, kept blocks):
//   625 of 25 36.5 / 37.1 (20 %, 50 %)    576 of 24 65.0 / 59.5 (75, 50) 37.9 / 29.8 (75, 10) 31.6 / 35.6 (20, 50)
//   500 of 125 213 / 182 (75, 50) 95.4 / 87.6 (30, 50)    480 of 40 83 / 76 (75, 50) 30.6 / 35.5 (10, 30)
// What it needs besides: partial results of two shares per CU, room in LDS for a row's list (the
// longest row is bounded by all keep bits where there are several requests), 32-bit copy offsets.
bool direct_pipe(const fo_attention_args& a, int num_cu) {
  const int64_t n_cand = direct_candidates(a);
  const int64_t nkv = a.max_nnz / (a.batch == 1 ? n_cand : a.symbol_heads), span = (nkv + 1) * kBlockKV * 2;
  const bool enough = a.is_full ? 8 * n_cand >= int64_t(13) * num_cu : 2 * n_cand >= int64_t(5) * num_cu;
  return a.logits_soft_cap <= 0.f && enough && nkv <= kMaxRowBlocksOneGroupDirect &&
         2 * num_cu <= kMaxShares && a.split_ws_bytes >= 2 * fo_sparse_fa_split_workspace_bytes() &&
         span * a.k_stride_n < (int64_t(1) << 32) && span * a.v_stride_n < (int64_t(1) << 32);
}

// Whether a share of the pipelined form has fewer rows than its table: a row costs kRowOverheadPipe at least, and a share
// is no longer than an even part of all cost, kOlderGain / 128 more, or four ninths of the longest row (of 3 and
// a part thirds 3 are made).  (At most 1.01 million keep bits on 256 CUs: a row is counted as one without kept blocks, and all keep
// bits as set, at the same time.)
bool direct_table_holds(int64_t n_cand, int64_t max_nnz, int num_cu) {
  const int64_t even = (max_nnz + kRowOverheadPipe * n_cand) / (2 * num_cu), longest = kMaxRowBlocksOneGroupDirect;
  return ((even + 2) * (128 + kOlderGain) / 128 / kRowOverheadPipe + 3 < kDirectShareRows &&
          (4 * longest / 9 + 2) / kRowOverheadPipe + 3 < kDirectShareRows);
}

// Whether the launch takes its rows straight from the symbols.
// Candidates that a workgroup's threads can go through at the top of a launch, and keep bits that every workgroup can
// afford to read (2^20 bits = 128 KB from L2: about as long as the scans).  Longer lists are worth a decode launch, which also
// sorts their rows by head, so that one head's K and V at a time are in an XCD's L2, and where they are enough rows for whole ones on
// two workgroups per CU (long_list) they run in the pipelined form as well.  The lists that only the pipelined form takes, decoded (and in
// the two-phase form) -> straight from the symbols, us per call (rows, blocks kept):
//   1440 of 60    736 -> 628 (all)
//   1720 of 43    635 -> 544 (all)
//   1840 of 46    750 -> 636 (all)  328 -> 276 (80, 50 %)  126 -> 93 (80, 10)  107 -> 90 (20, 50)  51.5 -> 39.6 (10, 20)
//   1824 of 76    1200 -> 1008      496 -> 427             147 -> 125          154 -> 134          61.1 -> 49.9
//   1920 of 128   2037 -> 1779      836 -> 731             221 -> 193          249 -> 215          78.0 -> 67.0
//   2040 of 85    1415 -> 1260      620 -> 531             175 -> 150          182 -> 164          65.7 -> 53.7
//   2040 of 170   2798 -> 2511      1188 -> 1032           289 -> 266          334 -> 299          94.7 -> 82.8
// (Decoded and in the pipelined form, whose queues have whole rows only, 1800 of 90 with 10 % of the rows take 78.7 in place of 63.4.)
bool direct_takes(const fo_attention_args& a, int variant) {
  const int num_cu = fo_num_cu();
  const int64_t n_cand = direct_candidates(a);
  return (a.dtype == FO_BF16 || a.dtype == FO_F16) && variant != 1 && n_cand >= 1 &&
         (n_cand <= direct_max_cand(0) ||
          (n_cand <= kDirectMost && variant == 0 && direct_pipe(a, num_cu) &&
           direct_table_holds(n_cand, a.max_nnz, num_cu))) &&
         a.max_nnz <= (1 << 20) && num_cu >= 16 && num_cu <= kMaxShares &&
         a.split_ws_bytes >= fo_sparse_fa_split_workspace_bytes();
}

}  // namespace

namespace {

bool direct_serves(const fo_attention_args& a) {
  return direct_takes(a, g_variant.load(std::memory_order_relaxed)) && a.split_ws &&
         (reinterpret_cast<uintptr_t>(a.split_ws) & 15) == 0;
}

// Longer lists are promised to callers not to touch a workspace that other batches' launches may be using: they need one of their own.
bool direct_shares_workspace(const fo_attention_args& a) {
  return direct_candidates(a) <= (a.is_full ? kDirectSharedFull : kDirectShared);
}

int direct_run(const fo_attention_args& a);

}  // namespace

extern "C" int fo_sparse_attention_direct_serves(const void* args) {
  const fo_attention_args& a = *static_cast<const fo_attention_args*>(args);
  return direct_shares_workspace(a) && direct_serves(a);
}

extern "C" int64_t fo_sparse_attention_direct_own_bytes(const void* args) {
  const fo_attention_args& a = *static_cast<const fo_attention_args*>(args);
  return !direct_shares_workspace(a) && direct_serves(a) ? 2 * fo_sparse_fa_split_workspace_bytes() : 0;
}

extern "C" int fo_sparse_attention_direct_may_serve(int32_t n_blk, int32_t symbol_heads, int32_t batch, int64_t max_nnz,
                                                    int64_t split_ws_bytes, float logits_soft_cap) {
  fo_attention_args a{};  // (the rest at its most favourable)
  a.dtype = FO_BF16;
  a.n_blk = n_blk;
  a.symbol_heads = symbol_heads;
  a.batch = batch;
  a.max_nnz = max_nnz;
  a.split_ws_bytes = split_ws_bytes;
  a.logits_soft_cap = logits_soft_cap;
  return direct_takes(a, 0);
}

extern "C" int32_t fo_sparse_attention_direct_max_pairs(void) { return kDirectMost; }

extern "C" int fo_sparse_attention_direct(const void* args) {
  FO_REQUIRE(args, "sparse_attention: null pointer");
  return fo_sparse_attention_direct_serves(args) ? direct_run(*static_cast<const fo_attention_args*>(args)) : FO_NOT_DIRECT;
}

extern "C" int fo_sparse_attention_direct_own(const void* args) {
  FO_REQUIRE(args, "sparse_attention: null pointer");
  return fo_sparse_attention_direct_own_bytes(args) ? direct_run(*static_cast<const fo_attention_args*>(args)) : FO_NOT_DIRECT;
}

namespace {

int direct_run(const fo_attention_args& a) {
  const int64_t n_cand = direct_candidates(a);
  FO_REQUIRE(a.q && a.k && a.v && a.o && a.qo_indptr && a.kv_indptr && a.blk_req && a.blk_qb && a.sched,
             "sparse_attention: null pointer");
  FO_REQUIRE(a.is_full || (a.info && a.kv_info && a.info_indptr && a.kv_info_indptr), "sparse_attention: null symbols");
  FO_REQUIRE(a.num_kv_heads > 0 && a.num_heads % a.num_kv_heads == 0, "sparse_attention: bad head counts");
  FO_REQUIRE(a.logits_soft_cap >= 0.f && a.logits_soft_cap < __builtin_inff(),
             "sparse_attention: logits_soft_cap must be a finite value >= 0 (0: no cap)");
  const int64_t strides[8] = {a.q_stride_n, a.q_stride_h, a.k_stride_n, a.k_stride_h,
                              a.v_stride_n, a.v_stride_h, a.o_stride_n, a.o_stride_h};
  for (int i = 0; i < 8; ++i)
    FO_REQUIRE(strides[i] % 8 == 0 && strides[i] > 0,
               "sparse_fa: strides must be positive multiples of 16 bytes (128-bit accesses)");
  FO_REQUIRE(a.q_stride_n < (int64_t(1) << 23) && a.k_stride_n < (int64_t(1) << 23) && a.v_stride_n < (int64_t(1) << 23),
             "sparse_fa: q/k/v token strides must be below 2^23 elements (32-bit tile offsets)");
  for (const void* ptr : {a.q, a.k, a.v, static_cast<const void*>(a.o)})
    FO_REQUIRE((reinterpret_cast<uintptr_t>(ptr) & 15) == 0, "sparse_fa: q/k/v/o must be 16-byte aligned");
  FaParams p{};
  p.q = a.q; p.k = a.k; p.v = a.v; p.o = a.o; p.lse = a.lse;
  p.q_sn = a.q_stride_n; p.q_sh = a.q_stride_h; p.k_sn = a.k_stride_n; p.k_sh = a.k_stride_h;
  p.v_sn = a.v_stride_n; p.v_sh = a.v_stride_h; p.o_sn = a.o_stride_n; p.o_sh = a.o_stride_h;
  p.qo_indptr = a.qo_indptr; p.kv_indptr = a.kv_indptr; p.sched = a.sched;
  p.split_ws = static_cast<float*>(a.split_ws);
  p.num_heads = a.num_heads;
  const bool packed = a.gqa_packed && a.num_heads != a.num_kv_heads;
  p.kv_group = packed ? 1 : a.num_heads / a.num_kv_heads;
  p.gqa_pack = packed ? a.num_heads / a.num_kv_heads : 0;
  p.sm_scale_log2 = a.sm_scale * 1.44269504088896340736f;
  p.info = a.info; p.kv_info = a.kv_info; p.info_indptr = a.info_indptr; p.kv_info_indptr = a.kv_info_indptr;
  p.blk_req = a.blk_req; p.blk_qb = a.blk_qb;
  p.n_blk = a.n_blk; p.batch = a.batch; p.symbol_heads = a.symbol_heads; p.is_full = a.is_full;
  p.zero_skipped = a.zero_skipped && !a.is_full;
  if (!a.is_full && (a.keep_info || a.keep_kv_info || a.keep_indptr)) {
    FO_REQUIRE(a.keep_info && a.keep_kv_info && a.keep_indptr, "sparse_attention: null pointer");
    p.keep_info = a.keep_info; p.keep_kv_info = a.keep_kv_info;
    p.info_bytes = a.info_bytes; p.kv_info_bytes = a.kv_info_bytes;
  } else {
    p.kv_info_bytes = a.kv_info_bytes > 0 ? a.kv_info_bytes : INT32_MAX;
  }
  p.keep_indptr = a.keep_indptr;
  hipStream_t s = static_cast<hipStream_t>(a.stream);
  const bool bf16 = a.dtype == FO_BF16;
  if (a.logits_soft_cap > 0.f) {
    p.cap_log2 = a.logits_soft_cap * 1.44269504088896340736f;
    p.sm_scale_log2 = 2.f * 1.44269504088896340736f * a.sm_scale / a.logits_soft_cap;
    if (packed)
      return bf16 ? launch<__bf16, false, false, false, 2, false, true, true, true>(p, n_cand, s)
                  : launch<_Float16, false, false, false, 2, false, true, true, true>(p, n_cand, s);
    return bf16 ? launch<__bf16, false, false, false, 2, false, false, true, true>(p, n_cand, s)
                : launch<_Float16, false, false, false, 2, false, false, true, true>(p, n_cand, s);
  }
  if (n_cand > direct_max_cand(0)) {
    auto many = [&](auto per) {
      constexpr int kPer = decltype(per)::value;
      if (packed)
        return bf16 ? launch<__bf16, false, false, false, 1, true, true, false, true, false, kPer>(p, n_cand, s)
                    : launch<_Float16, false, false, false, 1, true, true, false, true, false, kPer>(p, n_cand, s);
      return bf16 ? launch<__bf16, false, false, false, 1, true, false, false, true, false, kPer>(p, n_cand, s)
                  : launch<_Float16, false, false, false, 1, true, false, false, true, false, kPer>(p, n_cand, s);
    };
    return n_cand <= direct_max_cand(7) ? many(std::integral_constant<int, 7>{}) : many(std::integral_constant<int, 8>{});
  }
  if (direct_pipe(a, fo_num_cu())) {
    if (packed)
      return bf16 ? launch<__bf16, false, false, false, 1, true, true, false, true>(p, n_cand, s)
                  : launch<_Float16, false, false, false, 1, true, true, false, true>(p, n_cand, s);
    return bf16 ? launch<__bf16, false, false, false, 1, true, false, false, true>(p, n_cand, s)
                : launch<_Float16, false, false, false, 1, true, false, false, true>(p, n_cand, s);
  }
  if (packed)
    return bf16 ? launch<__bf16, false, false, false, 2, false, true, false, true>(p, n_cand, s)
                : launch<_Float16, false, false, false, 2, false, true, false, true>(p, n_cand, s);
  return bf16 ? launch<__bf16, false, false, false, 2, false, false, false, true>(p, n_cand, s)
              : launch<_Float16, false, false, false, 2, false, false, false, true>(p, n_cand, s);
}

}  // namespace
