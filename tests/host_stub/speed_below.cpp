// Host driver of QuickSpeedBelow and SpeedBelow (fvs_godunov_bound.hpp): reads n pairs of 2D
// conservative states (rho, m0, m1, E each side) and a speed a pair, doubles
// in component-major order, from the file argv[1]; prints how many pairs each
// test certifies to stay below their own speed, and below 1.05 and 2 times it.
// argv[2]: Newton iteration cap, argv[3]: gamma.
#include <cmath>
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(x))
#include "fvs_godunov_bound.hpp"

#include <cstdio>
#include <cstdlib>
#include <vector>

int main(int argc, char** argv) {
  std::FILE* f = std::fopen(argv[1], "rb");
  std::fseek(f, 0, SEEK_END);
  const long n = std::ftell(f) / 72;
  std::rewind(f);
  std::vector<double> v(9 * n);
  if (std::fread(v.data(), 72, n, f) != static_cast<size_t>(n)) return 1;
  const double gamma = std::atof(argv[3]);
  const fvs::SpeedBound b = fvs::MakeSpeedBound(gamma, 1e-7, std::atoi(argv[2]));
  const fvs::Gas<double> g{gamma, 1.0 / (gamma - 1.0), gamma - 1.0};
  long count[2][3] = {};
  const double scale[3] = {1.0 - 0x1p-20, 1.05, 2.0};
  for (long i = 0; i < n; ++i) {
    double q[2][4];
    for (int k = 0; k < 8; ++k) q[k / 4][k % 4] = v[k * n + i];
    const auto L = fvs::MakeSpeedCell<2>(q[0], g), R = fvs::MakeSpeedCell<2>(q[1], g);
    for (int k = 0; k < 3; ++k) {
      const float F = static_cast<float>(v[8 * n + i] * scale[k]);
      count[0][k] += fvs::QuickSpeedBelow<2>(L, L.u[0], R, R.u[0], b, F);
      count[1][k] += fvs::SpeedBelow<2>(L, L.u[0], R, R.u[0], b, F);
    }
  }
  for (int t = 0; t < 2; ++t)
    std::printf("%ld %ld %ld\n", count[t][0], count[t][1], count[t][2]);
  return 0;
}
