// What the one-launch kernels of small systems share (fwd_small_kernel in
// nb_forward.hip, adj_small_kernel in nb_adjoint.hip): the workgroup, the
// sums over a row of 16 lanes, the targets per row.
#pragma once

#include <hip/hip_runtime.h>

namespace nb {

constexpr int kSmallBlock = 1024;
constexpr int kSmallLanes = 16;                         // source lanes per row
constexpr int kSmallStride = kSmallBlock / 64 * kSmallLanes; // sources per pass
constexpr int kSmallBatch = 4;

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                         0xf, 0xf, false));
}

// (s, c) stands for s - c.  TwoSum keeps the rounding of s + s' in c.
__device__ __forceinline__ void meet(float &s, float &c, float s2, float c2) {
  const float t = s + s2;
  const float b = t - s;
  const float err = (s - (t - b)) + (s2 - b);
  c = (c + c2) - err;
  s = t;
}

template <bool KAHAN, int CTRL>
__device__ __forceinline__ void row_step(float &s, float &c) {
  if constexpr (KAHAN)
    meet(s, c, dpp<CTRL>(s), dpp<CTRL>(c));
  else
    s = s + dpp<CTRL>(s);
}

// Sum over a row of 16 lanes, in every lane of it (row_ror 8, 4, 2, 1).
template <bool KAHAN>
__device__ __forceinline__ void row_sum(float &s, float &c) {
  row_step<KAHAN, 0x128>(s, c);
  row_step<KAHAN, 0x124>(s, c);
  row_step<KAHAN, 0x122>(s, c);
  row_step<KAHAN, 0x121>(s, c);
}

// Targets per row of the one-launch shape: as few as leave one workgroup for
// each of the 256 CUs.  1 / 2 / 4 targets, us: n = 1000 3.4 / 3.6 / 4.3, 1500
// 4.7 / 4.3 / 5.4, 2000 5.1 / 4.6 / 5.8, 3000 8.1 / 7.7 / 7.5, 4000 11.7 / 9.2
// / 8.9.
inline int small_targets(int n) { return n <= 1024 ? 1 : n <= 2048 ? 2 : 4; }

} // namespace nb
