// Neighbour exchange between the lanes of a wave, and the blocks of kernels
// that advance a grid several sweeps per launch.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

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
template <int CTRL>
__device__ __forceinline__ float dpp_or(float edge, float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(x), CTRL,
                                                    0xF, 0xF, false));
}
template <class C>
__device__ __forceinline__ C lane_from_left_or(C edge, C x) {
  return dpp_or<0x138>(edge, x);
}
template <class C>
__device__ __forceinline__ C lane_from_right_or(C edge, C x) {
  return dpp_or<0x130>(edge, x);
}

// A workgroup barrier that orders LDS only: with __syncthreads the waves would
// also wait for every global load and store in flight, which the other threads
// do not touch.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A direction of a grid split into blocks that advance several sweeps per
// launch: n interior points, regions of `width` points held by a workgroup,
// halos of `depth` points where a region ends inside the grid and none where
// it ends with it.  Block t of `count` has its region's first interior point
// at grid index origin (from 1) and owns the region's points [lo, hi); the
// last region is shifted back to end with the grid.
struct Span {
  int origin, lo, hi;
  int width, first, last;  // first, last: whether the region ends with the grid
  // The sweeps, counted from 1, from which on none of the region's points
  // [from, to) is needed: a halo is valid for one cell less each sweep.
  __device__ __forceinline__ int useful(int from, int to) const {
    return min(first ? INT_MAX : to, last ? INT_MAX : width - from);
  }
};
__host__ __device__ inline int span_count(int n, int width, int depth) {
  const int out = width - 2 * depth;
  return n <= width ? 1 : (n - 2 * depth + out - 1) / out;
}
__device__ __forceinline__ Span span_of(int t, int count, int n, int width, int depth) {
  const int out = width - 2 * depth;
  const int o = t == count - 1 ? max(n - width, 0) : t * out;
  return {1 + o, (t == 0 ? 0 : t * out + depth) - o,
          (t == count - 1 ? n : (t + 1) * out + depth) - o, width, t == 0, t == count - 1};
}

}  // namespace npbx
