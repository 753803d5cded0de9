// The Jacobi rotation of the pair solves on the host, its reciprocal square
// root a unit in the last place off at random (what the instruction may be).
// Prints the largest errors over pairs of several kinds: the element that is
// left, over r; c^2 + s^2 - 1; and t against s / c.
#include <cmath>
#include <cstdio>
#include <random>

#define __device__
#define __forceinline__ inline

static std::mt19937_64 rng(12345);
static float rsq_near(float x) {
  const float y = (float)(1.0 / std::sqrt((double)x));
  const int k = (int)(rng() % 3) - 1;
  return k == 0 ? y : std::nextafterf(y, k > 0 ? INFINITY : 0.0f);
}
#define __builtin_amdgcn_rsqf rsq_near
using std::copysign;
using std::fma;
#include "../../mopac_gpu_amd/csrc/jacobi_rotation.h"

typedef long double Wide;

int main() {
  std::normal_distribution<double> g;
  std::uniform_real_distribution<double> u(-12.0, 0.0);
  Wide left = 0, length = 0, tangent = 0;
  for (int i = 0; i < 1000000; ++i) {
    double app = g(rng), aqq = g(rng), apq = g(rng);
    if (i % 3 == 1) apq *= std::pow(10.0, u(rng));
    if (i % 3 == 2) {
      aqq = app + (aqq - app) * std::pow(10.0, u(rng));
      apq *= std::pow(10.0, u(rng));
    }
    if (i % 7 == 0) app *= 1e3, aqq *= 1e3;
    double c, s, t;
    mhip::rotation_of(app, aqq, apq, c, s, t);
    const Wide d = (Wide)(aqq - app), C = c, S = s;
    const Wide r = std::sqrt(d * d + 4 * (Wide)apq * apq);
    left = std::fmax(left, std::fabs((C * C - S * S) * apq - C * S * d) / r);
    length = std::fmax(length, std::fabs(C * C + S * S - 1));
    if (s != 0) tangent = std::fmax(tangent, std::fabs(t * C / S - 1));
  }
  std::printf("%.3Le %.3Le %.3Le\n", left, length, tangent);
  return 0;
}
