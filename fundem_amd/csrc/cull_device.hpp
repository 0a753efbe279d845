// Conservative tests shared by the list builds and the narrow phase.
#pragma once
#include "fdm_device.hpp"

namespace fdm {

// Relative margin of every reach: a unit quaternion stored in FP32 scales
// vectors by up to 1 +- 2.4e-7.
constexpr double kReach = 1.0 + 1e-5;

// True when the ball (local, reach) misses the SDF box of t (target frame).
__device__ __forceinline__ bool outsideBox(V3 local, double reach, const fdm_template& t) {
  const double h = 1.0 / t.invSpacing;
  double d2 = 0.0;
  const double lo[3] = {t.origin[0], t.origin[1], t.origin[2]};
  const double p[3] = {local.x, local.y, local.z};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double hi = lo[a] + h * (double)(t.size[a] - 1);
    const double m = 1e-6 * (hi - lo[a]);
    double e = 0.0;
    if (p[a] < lo[a] - m) e = lo[a] - m - p[a];
    else if (p[a] > hi + m) e = p[a] - hi - m;
    d2 += e * e;
  }
  const double r = reach * kReach;
  return d2 > r * r;
}

// Clamped cell range of the box [c - r, c + r] (monotone in each coordinate).
__device__ __forceinline__ void cellRange(V3 c, double r, const fdm_grid& g, I3& lo, I3& hi) {
  lo = clampedCell(vsub(c, {r, r, r}), g);
  hi = clampedCell(vadd(c, {r, r, r}), g);
}
// True when no point within `reach` of `local` (target frame) can have
// phi <= 0: the point is inside the SDF box and phi - Lip*reach is positive
// beyond a relative margin.
__device__ __forceinline__ bool lipschitzClear(V3 local, double reach, const fdm_template& t,
                                               const float* sdf) {
  Sample s;
  if (!sampleSDF(local, t, sdf, s)) return false;
  const double phi = trilinear(s.x, s.y, s.z, s.c);
  const double lr = t.lipschitz * reach;
  return phi - lr > 1e-6 * (fabs(phi) + lr);
}

}  // namespace fdm
