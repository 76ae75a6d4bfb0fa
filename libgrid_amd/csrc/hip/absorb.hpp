// The absorbing boundary's amplitude (reference src/grid_wf.c, grid_wf_absorb).
#pragma once
#include <hip/hip_runtime.h>

namespace lg {

// one axis's share: the distance outside [lo, hi] over the lower bound (on both sides)
__device__ __forceinline__ double absorb_part(long i, long lo, long hi) {
  return i < lo ? (double)(lo - i) / (double)lo : i > hi ? (double)(i - hi) / (double)lo : 0.0;
}
// the shares of x, y and z summed in this order, times 2/3, capped at 1
__device__ __forceinline__ double absorb_sum(double x, double y, double z) {
  const double t = ((x + y) + z) * (2.0 / 3.0);
  return t > 1.0 ? 1.0 : t;
}

}  // namespace lg
