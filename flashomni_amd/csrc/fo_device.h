// Device helpers that more than one kernel file uses.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace fo {

// Inclusive prefix sum over the 64 lanes of a wavefront.  Rows of 16 lanes by data-parallel lane
// shifts (vector ALU speed; lanes shifted in from outside a row read zero), then the three row
// totals through scalar registers.  (Lane shuffles go through the LDS unit, which the sixteen
// wavefronts of a scan workgroup share: 12 per value made that unit the scan's bottleneck.)
__device__ __forceinline__ int32_t wave_scan(int32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);  // row_shr:8
  const int32_t t0 = __builtin_amdgcn_readlane(v, 15), t1 = __builtin_amdgcn_readlane(v, 31),
                t2 = __builtin_amdgcn_readlane(v, 47);
  const int row = (threadIdx.x & 63) >> 4;
  return v + (row >= 1 ? t0 : 0) + (row >= 2 ? t1 : 0) + (row >= 3 ? t2 : 0);
}

// The largest of the 64 lanes' values, none of them negative (lanes shifted in from outside a row read zero), in the
// same way.
__device__ __forceinline__ int32_t wave_max(int32_t v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));  // row_shr:1
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));  // row_shr:2
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));  // row_shr:4
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));  // row_shr:8
  return max(max(__builtin_amdgcn_readlane(v, 15), __builtin_amdgcn_readlane(v, 31)),
             max(__builtin_amdgcn_readlane(v, 47), __builtin_amdgcn_readlane(v, 63)));
}

}  // namespace fo
