// Neighbour exchange between the lanes of a wave.
#pragma once

#include <hip/hip_runtime.h>

namespace npbx {

// Full-wave DPP shifts (wave_shr:1, wave_shl:1): lane l receives lane l-1's
// (from_left) or lane l+1's (from_right) value; lanes 0 and 63 receive 0.
__device__ __forceinline__ int dpp_shr(int x) {
  return __builtin_amdgcn_update_dpp(0, x, 0x138, 0xF, 0xF, true);
}
__device__ __forceinline__ int dpp_shl(int x) {
  return __builtin_amdgcn_update_dpp(0, x, 0x130, 0xF, 0xF, true);
}
__device__ __forceinline__ float lane_from_left(float x) {
  return __int_as_float(dpp_shr(__float_as_int(x)));
}
__device__ __forceinline__ float lane_from_right(float x) {
  return __int_as_float(dpp_shl(__float_as_int(x)));
}
__device__ __forceinline__ double lane_from_left(double x) {
  return __hiloint2double(dpp_shr(__double2hiint(x)), dpp_shr(__double2loint(x)));
}
__device__ __forceinline__ double lane_from_right(double x) {
  return __hiloint2double(dpp_shl(__double2hiint(x)), dpp_shl(__double2loint(x)));
}


// The same with the value lane 0 (or lane 63) takes instead of 0: its own
// entry of `edge`.
template <int CTRL>
__device__ __forceinline__ double dpp_or(double edge, double x) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(x), CTRL, 0xF, 0xF, false),
      __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(x), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ double lane_from_left_or(double edge, double x) {
  return dpp_or<0x138>(edge, x);
}
__device__ __forceinline__ double lane_from_right_or(double edge, double x) {
  return dpp_or<0x130>(edge, x);
}

}  // namespace npbx
