// Steps within one wavefront, shared by the kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace hfx {

// LDS written by lanes of this wavefront before is read by others after.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// value of v in another lane of the row of 16 (DPP control CTRL); ZERO: 0 from
// outside the row (the controls that stay inside it need no such rule)
template <int CTRL, bool ZERO>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, ZERO);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, ZERO);
  return __hiloint2double(hi, lo);
}

// value of v in lane l, the same for all
__device__ __forceinline__ double lane_value(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// largest v of each row of 16 lanes, in every lane of it: butterflies on
// quad_perm, row_half_mirror and row_mirror
__device__ __forceinline__ double row_max(double v) {
  v = fmax(v, dpp_move<0xB1, false>(v));
  v = fmax(v, dpp_move<0x4E, false>(v));
  v = fmax(v, dpp_move<0x141, false>(v));
  return fmax(v, dpp_move<0x140, false>(v));
}

}  // namespace hfx
