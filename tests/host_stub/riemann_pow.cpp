// Host check of PowPos (fvs_riemann.hpp) against extended-precision powers:
// prints the largest error in units in the last place over the ratios and
// exponents of the exact Riemann solver (below 1, and those of fans).
#define __builtin_amdgcn_logf(x) std::log2(x)
#define __builtin_amdgcn_exp2f(x) std::exp2(x)
#include <cmath>
#include "fvs_riemann.hpp"

#include <cstdio>
#include <random>

int main() {
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> uni(0.0, 1.0);
  const double g[4] = {1.4, 5.0 / 3.0, 1.1, 1.3};
  double worst[2] = {0.0, 0.0};  // exponents below 1, fans
  for (int i = 0; i < 2000000; ++i) {
    const double gm = g[i & 3], gm1 = gm - 1.0;
    const double es[4] = {0.5 * gm1 / gm, 1.0 / gm, 2.0 / gm1, 2.0 * gm / gm1};
    const double e = es[(i >> 2) & 3];
    double x;
    switch ((i >> 4) & 3) {
    case 0: x = uni(rng); break;                               // rarefactions
    case 1: x = std::exp(-14.0 * uni(rng)); break;             // strong ones
    case 2: x = 1.0 - std::ldexp(uni(rng), -(i >> 6) % 52); break;  // weak ones
    default: x = std::ldexp(0.5 + uni(rng), ((i >> 6) % 40) - 20);  // any
    }
    if (!(x > 0.0)) continue;
    const long double want = powl(static_cast<long double>(x), static_cast<long double>(e));
    const double got = fvs::PowPos(x, e);
    const double ulp = std::nextafter(static_cast<double>(want), 1e308) - static_cast<double>(want);
    const double err = static_cast<double>(fabsl(got - want)) / ulp;
    double& w = worst[e < 1.0 ? 0 : 1];
    if (err > w) w = err;
  }
  // edges: one, the smallest normal and denormal numbers, and PowState's
  // zero, infinity, negative and NaN
  const double e = 1.0 / 7.0;
  int bad = fvs::PowPos(1.0, e) != 1.0;
  for (double x : {0x1p-1022, 0x1p-1074, 0x1.8p-1060, 0x1p-1000, 0x1.fffffffffffffp1023}) {
    const double want = static_cast<double>(powl(x, e));
    bad += !(std::fabs(fvs::PowPos(x, e) / want - 1.0) < 3e-16);
  }
  bad += fvs::PowState(0.0, e) != 0.0;
  bad += !std::isinf(fvs::PowState(HUGE_VAL, e));
  bad += !std::isnan(fvs::PowState(-1.0, e)) + !std::isnan(fvs::PowState(NAN, e));
  // negative numbers have whole powers only (and infinite ones any)
  bad += fvs::PowState(-2.0, 3.0) != -8.0 || fvs::PowState(-2.0, 4.0) != 16.0;
  bad += !std::isnan(fvs::PowState(-2.0, 5.000000000000001));
  bad += fvs::PowState(-HUGE_VAL, 3.0) != -HUGE_VAL || fvs::PowState(-HUGE_VAL, 5.5) != HUGE_VAL;
  std::printf("%.3f %.3f %d\n", worst[0], worst[1], bad);
  return 0;
}
