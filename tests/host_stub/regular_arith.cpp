// RegularArith (fvs_physics.hpp) on the host, from reciprocal and reciprocal
// square root estimates wrong by up to 2^-24 of their values: prints how many
// reciprocals, quotients and roots are not the correctly rounded ones.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <random>
#undef __builtin_amdgcn_rcp
#undef __builtin_amdgcn_rsq
#undef __builtin_amdgcn_div_fixup
#undef __builtin_amdgcn_class
static std::mt19937_64 rng(11);
static double Off() { return 1.0 + std::uniform_real_distribution<double>(-0x1p-24, 0x1p-24)(rng); }
static double Rcp(double b) { return (1.0 / b) * Off(); }
static double Rsq(double x) { return (1.0 / std::sqrt(x)) * Off(); }
static double Fixup(double q, double b, double a) {
  return (a == 0.0 || b == 0.0 || !std::isfinite(a) || !std::isfinite(b)) ? a / b : q;
}
#define __builtin_amdgcn_rcp(x) Rcp(x)
#define __builtin_amdgcn_rsq(x) Rsq(x)
#define __builtin_amdgcn_div_fixup(q, b, a) Fixup(q, b, a)
#define __builtin_amdgcn_class(x, m) ((x) == 0.0 || (x) == INFINITY)
#include "fvs_physics.hpp"

int main() {
  using A = fvs::RegularArith<double>;
  std::uniform_real_distribution<double> m(1.0, 2.0);
  std::uniform_int_distribution<int> e(-200, 200), few(1, 300), kind(0, 3);
  long bad[3] = {0, 0, 0};
  for (long i = 0; i < 3000000; ++i) {
    double s = m(rng);
    switch (kind(rng)) {
    case 0: s = 2.0 - few(rng) * 0x1p-52; break;                 // next to 2
    case 1: s = 1.0 + few(rng) * 0x1p-52; break;                 // next to 1
    case 2: s = 2.0 - std::ldexp(m(rng), -1 - (i % 52)); break;  // between
    }
    if (i < 4) s = 2.0 - 0x1p-52;
    if (i == 4) s = (0x1p53 - 0x1p27 + 1.0) * 0x1p-52;  // 1 / s just below a tie
    const double b = std::ldexp(s, e(rng)) * ((i & 1) ? -1.0 : 1.0);
    double a = std::ldexp(m(rng), e(rng));
    if (i & 2) a = std::ldexp(2.0 - few(rng) * 0x1p-52, e(rng));
    if (i & 4) a = 0x1.6666666666663p+1;
    const A::Inv y = A::inv(b);
    if (y.y != 1.0 / b) ++bad[0];
    if (A::div(a, y) != a / b) ++bad[1];
    const double x = std::fabs(b);
    if (A::sqrt(x) != std::sqrt(x)) ++bad[2];
  }
  if (A::quot(0.0, 3.0) != 0.0 || !std::isinf(A::quot(1.0, 0.0)) || !std::isnan(A::quot(0.0, 0.0)) ||
      A::sqrt(0.0) != 0.0 || !std::isinf(A::sqrt(INFINITY)) || !std::isnan(A::sqrt(-1.0)))
    ++bad[1];
  std::printf("%ld %ld %ld\n", bad[0], bad[1], bad[2]);
  return bad[0] + bad[1] + bad[2] != 0;
}
