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

// The same step for x > 0 (no charge on the point): one clamp fewer.
__device__ __forceinline__ double rsqrt_refine_pos(float seed, double x) {
  const double y = (double)seed;
  const double e = fma(-x, y * y, 1.0);
  return fma(0.5 * y, e, y);
}

// 1 / r of the interpolating and the one-launch kernels: returned for the
// potential (+inf at r = 0, not a number at r = inf; KEEP_NAN has none), and in
// re for the field:
// 0 for a charge beyond the FP32 range of r^2 (as an FP32 rsq of inf has it), at
// most rclamp under the r^2 >= 1e-6 floor (SOFT).  The 1 / r of a coordinate that
// is not a number stays one where KEEP_NAN (E alone on a grid), so that all three
// components are, and becomes the floor's otherwise: what the direct kernels give,
// whose E alone on a grid has no floor where no charge is near a point.  KEEP_NAN
// costs nothing: the select falls back to the seed itself instead of to 0, and
// the step needs no clamp for r = 0, whose NaN fmin turns into the floor's 1 / r.
// 101^3 x 30,000 charges with NaN turned into the floor 228 us, with this 226,
// with an FP64 comparison in place of fmin 234.
template <bool SOFT, bool KEEP_NAN>
__device__ __forceinline__ double pair_rsqrt(double r2, double rclamp, double& re) {
  const float seed = __builtin_amdgcn_rsqf((float)r2);
  if constexpr (SOFT && KEEP_NAN) {
    const double v = rsqrt_refine_pos(seed, r2);
    re = seed > 0.f ? fmin(v, rclamp) : (double)seed;
    return v;
  }
  const double v = rsqrt_refine(seed, r2);
  re = seed == 0.f ? 0.0 : v;
  if constexpr (SOFT) re = fmin(re, rclamp);
  return v;
}

// The floor's 1 / r.
__device__ __forceinline__ double pair_clamp() {
  return rsqrt_refine(__builtin_amdgcn_rsqf(1e-6f), (double)1e-6f);
}

}  // namespace cpet
