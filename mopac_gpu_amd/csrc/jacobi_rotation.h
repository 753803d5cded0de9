// The Jacobi rotation of one index pair.
#pragma once

namespace mhip {
namespace {

// Rotation by the smaller of the angles that zero apq in [[app, apq], [apq,
// aqq]]: with d = aqq - app, h = 2 apq and r = sqrt(d^2 + h^2), c^2 = (1 +
// |d| / r) / 2 and s = sign(d) h / (2 r c); t = s / c, and the diagonal after
// it is app - t apq, aqq + t apq.  c and s start in FP32 (a reciprocal square
// root is one instruction there), an FP64 step turns them by what they leave
// of apq, and they are scaled to c^2 + s^2 = 1 in FP64.  The turn is what is
// left over the levels' distance, whose reciprocal is FP32's 1 / r after a
// Newton step: with that 1 / r itself, good to 3e-7, 1e-13 r was left of an
// element that is then taken for zero.  Over 10^6 pairs 1.6e-16 r is left at
// most, 2.0e-16 with FP64 division and square roots throughout, and c^2 + s^2
// is 1 to 4e-16.
// Every round of a pair solve waits for this chain of 18 dependent operations;
// FP64 division and square roots take 100.  With apq and d both below 1e-15,
// far under any stopping threshold (they are absolute), nothing is turned.
__device__ __forceinline__ void rotation_of(double app, double aqq, double apq, double& c, double& sn,
                                            double& t) {
  const double d = aqq - app;
  const float df = (float)d, ad = fabsf(df), hh = (float)apq;
  const float r2 = fmaf(4.0f * hh, hh, ad * ad);
  const float rinv = __builtin_amdgcn_rsqf(r2);
  const float c2 = fmaf(0.5f * ad, rinv, 0.5f);
  const float cinv = __builtin_amdgcn_rsqf(c2);
  const bool none = r2 < 1.0e-30f;
  const float cf = none ? 1.0f : c2 * cinv, sf = none ? 0.0f : copysignf(1.0f, df) * hh * rinv * cinv;
  const double c0 = (double)cf, s0 = (double)sf;
  const double p = fma(c0, c0, -s0 * s0), q = c0 * s0;
  // the off-diagonal element and the levels' distance after that rotation
  const double left = fma(p, apq, -q * d), dist = fma(p, d, q * (4.0 * apq));
  // left / dist, 1 / dist by a Newton step from FP32's 1 / r
  const double ri = (double)(none ? 0.0f : copysignf(rinv, df));
  const double turn = left * ri * fma(-dist, ri, 2.0);
  const double c1 = fma(-turn, s0, c0), s1 = fma(turn, c0, s0);
  const double e = fma(-c1, c1, fma(-s1, s1, 1.0));
  const double corr = fma(e, fma(e, 0.375, 0.5), 1.0);
  c = c1 * corr;
  sn = s1 * corr;
  // s / c, 1 / c by a third-order step from FP32's
  const double ci = none ? 1.0 : (double)cinv, ec = fma(-c, ci, 1.0), t1 = sn * ci;
  t = fma(t1, fma(ec, ec, ec), t1);
}

}  // namespace
}  // namespace mhip
