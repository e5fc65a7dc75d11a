// packbits / segment_packbits for gfx950: eight bool bytes are gathered into one output byte with a
// multiply (aligned packbits: 64 bools per lane, four 16-byte loads and one 8-byte store);
// HBM-bound (n bytes read, n/8 written).
// Semantics: numpy.packbits per segment (reference: include/flashomni/quantization.cuh:39-83).
#include "fo_common.h"

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ uint8_t pack8(uint64_t bools, int little) {
  // normalise every byte to 0/1
  uint64_t nz = bools | (bools >> 4);
  nz |= nz >> 2;
  nz |= nz >> 1;
  nz &= 0x0101010101010101ull;
  // byte j (memory order) carries element j.  little: bit j.  big: bit 7-j.
  const uint64_t mul = little ? 0x0102040810204080ull : 0x8040201008040201ull;
  return static_cast<uint8_t>((nz * mul) >> 56);
}

__device__ __forceinline__ uint64_t load8_guarded(const uint8_t* p, int64_t remaining) {
  // `remaining` bytes are readable at p; missing ones read as 0
  if (remaining >= 8 && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
    return *reinterpret_cast<const uint64_t*>(p);
  }
  uint64_t v = 0;
  const int n = remaining < 8 ? static_cast<int>(remaining) : 8;
  for (int j = 0; j < n; ++j) v |= static_cast<uint64_t>(p[j]) << (8 * j);
  return v;
}

// kVec: x is 16-byte and y 8-byte aligned: a lane turns 64 bools (four 16-byte loads, all in flight
// together) into one 8-byte store; the last n % 64 bools go the byte-wise way.
template <bool kVec>
__global__ void __launch_bounds__(kThreads) packbits_kernel(const uint8_t* __restrict__ x,
                                                            int64_t n, int little,
                                                            uint8_t* __restrict__ y) {
  typedef __attribute__((ext_vector_type(2))) uint64_t u64x2;
  const int64_t nbytes = (n + 7) >> 3;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  const int64_t tid = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  int64_t done = 0;  // output bytes covered by the vector part
  if constexpr (kVec) {
    const int64_t nvec = n >> 6;
    for (int64_t v = tid; v < nvec; v += stride) {
      const u64x2* src = reinterpret_cast<const u64x2*>(x + v * 64);
      const u64x2 a = src[0], b = src[1], c = src[2], d = src[3];
      const uint64_t out = static_cast<uint64_t>(pack8(a[0], little)) | static_cast<uint64_t>(pack8(a[1], little)) << 8 |
                           static_cast<uint64_t>(pack8(b[0], little)) << 16 | static_cast<uint64_t>(pack8(b[1], little)) << 24 |
                           static_cast<uint64_t>(pack8(c[0], little)) << 32 | static_cast<uint64_t>(pack8(c[1], little)) << 40 |
                           static_cast<uint64_t>(pack8(d[0], little)) << 48 | static_cast<uint64_t>(pack8(d[1], little)) << 56;
      *reinterpret_cast<uint64_t*>(y + v * 8) = out;
    }
    done = nvec * 8;
  }
  for (int64_t i = done + tid; i < nbytes; i += stride) {
    y[i] = pack8(load8_guarded(x + i * 8, n - i * 8), little);
  }
}

__global__ void __launch_bounds__(kThreads) segment_packbits_kernel(
    const uint8_t* __restrict__ x, const int32_t* __restrict__ in_indptr,
    const int32_t* __restrict__ out_indptr, int little, uint8_t* __restrict__ y) {
  const int seg = blockIdx.y;
  const int64_t begin = in_indptr[seg];
  const int64_t n = in_indptr[seg + 1] - begin;
  const int64_t nbytes = (n + 7) >> 3;
  const int64_t out0 = out_indptr[seg];
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < nbytes;
       i += stride) {
    y[out0 + i] = pack8(load8_guarded(x + begin + i * 8, n - i * 8), little);
  }
}

// Segments with their output offsets worked out here: x holds n bools, segment i packs
// x[indptr[i] : indptr[i+1]] and begins at the next output byte.  Every workgroup takes the prefix sum of
// the segments' byte counts itself (at most kMaxScanSegments, one batch of loads and a scan), so there is
// no pass in front of this one; a lane then owns 8 output bytes.  Inside a segment that is 64 bools through
// four 16-byte loads of any alignment and one 8-byte store, otherwise byte by byte.  Bound by launch
// latency at the sizes of a mask (1.6 M bools of a 33 k token video layer: 2.6 us).  Workgroup 0 writes
// the output's indptr, and the total with the caller's ticket to `total` (pinned host memory, or null):
// the host reads the length there, and waits neither for a copy nor for the rest of the stream's work.
// An indptr that descends, leaves x or needs more than `capacity` bytes packs nothing: total = -1.
constexpr int kMaxScanSegments = 1024;
template <typename I>
__global__ void __launch_bounds__(kThreads) segment_packbits_scan_kernel(
    const uint8_t* __restrict__ x, int64_t n, const I* __restrict__ indptr, int num_segments, int little,
    uint8_t* __restrict__ y, int64_t capacity, int32_t* __restrict__ out_indptr, uint64_t* total, uint32_t ticket) {
  __shared__ int64_t s_begin[kMaxScanSegments + 1];
  __shared__ int32_t s_out[kMaxScanSegments + 1];
  __shared__ int64_t s_wave[kThreads / 64];
  __shared__ int s_bad;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) s_bad = 0;
  for (int i = tid; i <= num_segments; i += kThreads) s_begin[i] = indptr[i];
  __syncthreads();
  int64_t carry = 0;
  for (int base = 0; base < num_segments; base += kThreads) {
    const int i = base + tid;
    int64_t bytes = 0;
    if (i < num_segments) {
      const int64_t len = s_begin[i + 1] - s_begin[i];
      if (len < 0 || s_begin[i] < 0 || s_begin[i + 1] > n) s_bad = 1; else bytes = (len + 7) >> 3;
    }
    int64_t incl = bytes;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t up = __shfl_up(incl, d, 64);
      if (lane >= d) incl += up;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    int64_t before = carry;
    for (int w = 0; w < kThreads / 64; ++w) {
      if (w < wave) before += s_wave[w];
      carry += s_wave[w];
    }
    if (i < num_segments) s_out[i] = static_cast<int32_t>(before + incl - bytes);
    __syncthreads();
  }
  if (tid == 0) s_out[num_segments] = static_cast<int32_t>(carry);
  __syncthreads();
  const bool bad = s_bad != 0 || carry > capacity;
  if (blockIdx.x == 0) {
    if (!bad)
      for (int i = tid; i <= num_segments; i += kThreads) out_indptr[i] = s_out[i];
    if (tid == 0 && total)
      __hip_atomic_store(total, static_cast<uint64_t>(ticket) << 32 | static_cast<uint32_t>(bad ? -1 : static_cast<int32_t>(carry)),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (bad) return;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads * 8;
  for (int64_t o = (static_cast<int64_t>(blockIdx.x) * kThreads + tid) * 8; o < carry; o += stride) {
    int lo = 0, hi = num_segments;  // last segment that begins at or before output byte o
    while (hi - lo > 1) {
      const int mid = (lo + hi) / 2;
      if (s_out[mid] <= o) lo = mid; else hi = mid;
    }
    const uint8_t* src = x + s_begin[lo] + (o - s_out[lo]) * 8;
    if (src + 64 <= x + s_begin[lo + 1]) {
      uint64_t v[8], out = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) __builtin_memcpy(&v[2 * j], src + 16 * j, 16);
#pragma unroll
      for (int j = 0; j < 8; ++j) out |= static_cast<uint64_t>(pack8(v[j], little)) << (8 * j);
      *reinterpret_cast<uint64_t*>(y + o) = out;
      continue;
    }
    for (int64_t b = o; b < min(o + 8, carry); ++b) {
      while (lo + 1 < num_segments && s_out[lo + 1] <= b) ++lo;  // (empty segments share a byte offset)
      const int64_t at = s_begin[lo] + (b - s_out[lo]) * 8;
      y[b] = pack8(load8_guarded(x + at, s_begin[lo + 1] - at), little);
    }
  }
}

int grid_for(int64_t nbytes) {
  int64_t g = (nbytes + kThreads - 1) / kThreads;
  if (g < 1) g = 1;
  if (g > 256 * 16) g = 256 * 16;
  return static_cast<int>(g);
}

}  // namespace

extern "C" int fo_packbits(const uint8_t* x, int64_t n, int bitorder, uint8_t* y, void* stream) {
  FO_REQUIRE(bitorder == FO_BITORDER_BIG || bitorder == FO_BITORDER_LITTLE,
             "bitorder must be 'big' or 'little'");
  FO_REQUIRE(n >= 0, "packbits: negative length");
  if (n == 0) return FO_OK;
  FO_REQUIRE(x && y, "packbits: null pointer");
  const bool vec = n >= 64 && ((reinterpret_cast<uintptr_t>(x) & 15) | (reinterpret_cast<uintptr_t>(y) & 7)) == 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (vec) {
    packbits_kernel<true><<<grid_for((n + 63) / 64), kThreads, 0, s>>>(x, n, bitorder == FO_BITORDER_LITTLE, y);
  } else {
    packbits_kernel<false><<<grid_for((n + 7) / 8), kThreads, 0, s>>>(x, n, bitorder == FO_BITORDER_LITTLE, y);
  }
  FO_CHECK_LAUNCH();
  return FO_OK;
}

extern "C" int fo_segment_packbits(const uint8_t* x, const int32_t* in_indptr,
                                   const int32_t* out_indptr, int32_t num_segments, int bitorder,
                                   uint8_t* y, void* stream) {
  FO_REQUIRE(bitorder == FO_BITORDER_BIG || bitorder == FO_BITORDER_LITTLE,
             "bitorder must be 'big' or 'little'");
  FO_REQUIRE(num_segments >= 0 && num_segments <= 65535, "segment_packbits: bad segment count %d",
             num_segments);
  if (num_segments == 0) return FO_OK;
  FO_REQUIRE(in_indptr && out_indptr, "segment_packbits: null indptr");
  // segment lengths live on the device: use a fixed, generous x-grid and stride inside
  dim3 grid(num_segments == 1 ? 1024 : 64, num_segments);
  segment_packbits_kernel<<<grid, kThreads, 0, static_cast<hipStream_t>(stream)>>>(
      x, in_indptr, out_indptr, bitorder == FO_BITORDER_LITTLE, y);
  FO_CHECK_LAUNCH();
  return FO_OK;
}

extern "C" int fo_segment_packbits_scan(const uint8_t* x, int64_t n, const void* indptr, int indptr_int64,
                                        int32_t num_segments, int bitorder, uint8_t* y, int64_t capacity,
                                        int32_t* out_indptr, uint64_t* total, uint32_t ticket, void* stream) {
  FO_REQUIRE(bitorder == FO_BITORDER_BIG || bitorder == FO_BITORDER_LITTLE,
             "bitorder must be 'big' or 'little'");
  FO_REQUIRE(num_segments >= 1 && num_segments <= kMaxScanSegments && n >= 0 && capacity >= 0 &&
                 capacity < (int64_t(1) << 31),
             "segment_packbits: bad sizes (1 to %d segments)", kMaxScanSegments);
  FO_REQUIRE(indptr && out_indptr && (x || n == 0) && (y || capacity == 0), "segment_packbits: null pointer");
  FO_REQUIRE((reinterpret_cast<uintptr_t>(y) & 7) == 0, "segment_packbits: y must be 8-byte aligned");
  const int grid = grid_for((capacity + 7) / 8), little = bitorder == FO_BITORDER_LITTLE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (indptr_int64) {
    segment_packbits_scan_kernel<<<grid, kThreads, 0, s>>>(x, n, static_cast<const int64_t*>(indptr), num_segments, little,
                                                           y, capacity, out_indptr, total, ticket);
  } else {
    segment_packbits_scan_kernel<<<grid, kThreads, 0, s>>>(x, n, static_cast<const int32_t*>(indptr), num_segments, little,
                                                           y, capacity, out_indptr, total, ticket);
  }
  FO_CHECK_LAUNCH();
  return FO_OK;
}
