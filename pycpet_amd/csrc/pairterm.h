// The FP64 pair term that the field kernels share.
#pragma once

#include <hip/hip_runtime.h>

namespace cpet {

// One Newton-Raphson step in FP64 from an FP32 estimate of 1/sqrt(x):
// relative error ~1e-7 -> ~1e-14.  Clamping y*y keeps x == 0 (y = +inf)
// from producing 0*inf: the residual is then 1 and the result stays +inf.
__device__ __forceinline__ double rsqrt_refine(float seed, double x) {
  const double y = (double)seed;
  const double e = fma(-x, fmin(y * y, 1.7976931348623157e308), 1.0);
  return fma(0.5 * y, e, y);
}

// 1 / r of the interpolating and the one-launch kernels: for the potential
// (+inf at r = 0, not a number at r = inf), and in ye for the field, where a
// charge beyond the FP32 range of r^2 adds 0 (as an FP32 rsq of inf does).
__device__ __forceinline__ double pair_rsqrt(double r2, double& ye) {
  const float seed = __builtin_amdgcn_rsqf((float)r2);
  const double v = rsqrt_refine(seed, r2);
  ye = seed == 0.f ? 0.0 : v;
  return v;
}

// ye under the r^2 >= 1e-6 floor (SOFT).  The 1 / r of a coordinate that is
// not a number stays one where KEEP_NAN (E alone on a grid), so that all three
// components are, and becomes the floor's otherwise: what the direct kernels
// give, whose E alone on a grid has no floor where no charge is near a point.
template <bool SOFT, bool KEEP_NAN>
__device__ __forceinline__ double pair_floor(double ye, double rclamp) {
  if constexpr (!SOFT) return ye;
  return KEEP_NAN ? (ye > rclamp ? rclamp : ye) : fmin(ye, rclamp);
}

}  // namespace cpet
