// Exact Riemann solver of the perfect gas on the device (FP64).
//
// Follows ExactRiemannSolver<PerfectGas<Dim>> operation for operation:
//   ComputeMiddleState   src/equations/perfect_gas/ExactRiemannSolver.hpp:34-97
//   NewtonIteration      include/fub/NewtonIteration.hpp:28-52
//   ComputeSignals       src/equations/perfect_gas/ExactRiemannSolver.hpp:105-148
//   SolveRiemannProblem  src/equations/perfect_gas/ExactRiemannSolver.hpp:204-353
//   Godunov flux / CFL   include/fub/flux_method/GodunovMethod.hpp:130-170
// The exact solver forces the reference onto its sequential (scalar) code
// path (the array ComputeSignals throws), so kinetic energies here use the
// scalar reduction order (m0^2 + m1^2) + m2^2.  Powers, quotients and roots
// can differ from the host's in the last bit, so these results agree with the
// CPU to rounding, not bit for bit.
//
// Arithmetic.  A face costs two to four evaluations of the pressure function,
// so the solver's sweeps are bound by FP64 instructions (VALU busy 74 to 77%),
// and the library's pow and the compiler's division and square root sequences
// were most of them.  Here
// powers are PowPos below, quotients and roots are NearArith (nearest or its
// neighbour), and an evaluation runs one branch a side (SolveMiddleState).
// First-order step on 384^3 strong-wave blocks: 42.7 -> 19.7 ms; per-face
// fluxes and stable dt of a 131 x 97 x 75 patch: 221 -> 131 us; the error of
// the states against 64-bit arithmetic stays at 1e-16 to 3e-16.
//
// States that are no gas (no or negative pressure, no density, infinities and
// NaNs) keep the numbers, infinities and NaNs of the reference's formulas:
// their sound speed is not positive and finite (IsGas), where the special
// results of the quotients are set (NearArith::fix; in every quotient it would
// cost 3% of a step).  Not kept are the results for densities and pressures
// beyond 1e150 or below 1e-150, whose products leave the range.
//
// Mixed form (MIXED = true): the same FP64 iteration; the sampled star
// density takes its power from the single-precision estimates,
// x^e = exp2(e log2 x).
#pragma once

#include "fvs_physics.hpp"

namespace fvs {

// Quotients and square roots for FP64 kernels that are held to a tolerance:
// a reciprocal (square root) from the hardware estimate (2^-24) refined by
// one Newton step, and one residual correction of the result, whose error
// beyond the final rounding is about 2^-45 units in the last place.  9
// instructions a quotient, 3 for each further one by the same denominator.
// A zero, infinite, subnormal or huge (above 2^1022) operand yields NaN; fix
// and sqrt set the results of zero and infinite ones.
struct NearArith {
  static __device__ __forceinline__ double inv(double b) {
    const double y = __builtin_amdgcn_rcp(b);
    return __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
  }
  // a / b with y = inv(b)
  static __device__ __forceinline__ double div(double a, double b, double y) {
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-q, b, a), y, q);
  }
  static __device__ __forceinline__ double quot(double a, double b) { return div(a, b, inv(b)); }
  // q, the quotient div(a, b, y), with the results of zero, infinite and NaN
  // operands set
  static __device__ __forceinline__ double fix(double q, double a, double b) {
    return __builtin_amdgcn_div_fixup(q, b, a);
  }
  static __device__ __forceinline__ double sqrt(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    double s = x * r;
    double h = 0.5 * r;
    const double e = __builtin_fma(-h, s, 0.5);
    s = __builtin_fma(s, e, s);
    h = __builtin_fma(h, e, h);
    s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
    return __builtin_amdgcn_class(x, 0x260) ? x : s;  // zeros, +infinity
  }
  // x^(-1/2) to about one unit in the last place: the estimate with one
  // third-order step, 1 / sqrt(1 - e) = 1 + e (1/2 + 3/8 e) + O(e^3).
  static __device__ __forceinline__ double rsqrt(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = __builtin_fma(-(x * y), y, 1.0);
    return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
  }
};

// x^e for positive finite x: 2^(e log2 x).  With x = 2^k m, m in
// [sqrt(1/2), sqrt(2)) and f = (m - 1) / (m + 1), log2 m = 2 / ln 2 atanh f
// = C f + f s Q(s), s = f^2; the quotient, the leading product and the sum
// with k keep their rounding errors (a log2 of about 2^-58), so the product
// with e does too.  k and m are taken from the high word by the addition that
// the FreeBSD and musl logarithms use.  2^r on [-1/2, 1/2] is a polynomial.  Both polynomials
// interpolate their function at Chebyshev nodes (relative errors below 1e-17).
// Result within 0.8 units in the last place for exponents below 1 and 1.1 for
// those of fans (against 80-bit powers, tests/test_riemann_pow.py), in about
// 75 instructions.
__device__ __forceinline__ double PowPos(double x, double e) {
  const bool tiny = x < 0x1p-1000;  // denormals too: scaled into the normal range
  const unsigned long long bits =
      static_cast<unsigned long long>(__double_as_longlong(tiny ? x * 0x1p200 : x));
  const unsigned int hi = static_cast<unsigned int>(bits >> 32) + (0x3ff00000u - 0x3fe6a09eu);
  const int k = static_cast<int>(hi >> 20) - (tiny ? 1223 : 1023);
  const unsigned long long mhi = (hi & 0xfffffu) + 0x3fe6a09eu;
  const double m =
      __longlong_as_double(static_cast<long long>((mhi << 32) | (bits & 0xffffffffull)));
  const double num = m - 1.0;
  const double den = m + 1.0;
  const double den_lo = m - (den - 1.0);
  const double y = NearArith::inv(den);
  const double f = num * y;
  const double f_lo = __builtin_fma(-f, den_lo, __builtin_fma(-f, den, num)) * y;
  const double s = f * f;
  double q = 0x1.afde0dd07fe15p-3;
  q = __builtin_fma(q, s, 0x1.c4ff2c46480e7p-3);
  q = __builtin_fma(q, s, 0x1.0c9e91c7d1b10p-2);
  q = __builtin_fma(q, s, 0x1.484b091a92bb1p-2);
  q = __builtin_fma(q, s, 0x1.a61762b534b6ep-2);
  q = __builtin_fma(q, s, 0x1.2776c50ef68f3p-1);
  q = __builtin_fma(q, s, 0x1.ec709dc3a0401p-1);
  const double C = 0x1.71547652b82fep+1, C_lo = 0x1.777d0ffda0d24p-55;  // 2 / ln 2
  const double l_hi = C * f;
  double l_lo = __builtin_fma(C, f, -l_hi);
  l_lo = __builtin_fma(C_lo, f, l_lo);
  l_lo = __builtin_fma(C, f_lo, l_lo);
  const double l_q = f * s * q;  // at most 1% of l_hi
  const double l = l_hi + l_q;
  l_lo += (l_hi - l) + l_q;
  const double kd = static_cast<double>(k);
  const double L = kd + l;
  const double L_lo = ((kd - L) + l) + l_lo;
  const double z = e * L;
  const double z_lo = __builtin_fma(e, L_lo, __builtin_fma(e, L, -z));
  const double n = __builtin_rint(z);
  const double r = z - n;
  double p = 0x1.e9d419696e0e9p-32;
  p = __builtin_fma(p, r, 0x1.e6065f532c950p-28);
  p = __builtin_fma(p, r, 0x1.b524fad88ed30p-24);
  p = __builtin_fma(p, r, 0x1.62bfd46781ef6p-20);
  p = __builtin_fma(p, r, 0x1.ffcbfc6712438p-17);
  p = __builtin_fma(p, r, 0x1.4309130975155p-13);
  p = __builtin_fma(p, r, 0x1.5d87fe78a526dp-10);
  p = __builtin_fma(p, r, 0x1.3b2ab6fba1dc6p-7);
  p = __builtin_fma(p, r, 0x1.c6b08d704a0c2p-5);
  p = __builtin_fma(p, r, 0x1.ebfbdff82c598p-3);
  // 2^(r + z_lo) = (1 + ln 2 r + r^2 p) (1 + ln 2 z_lo): the rounding error of
  // 1 + ln 2 r joins the small terms, which are added last
  const double ln2 = 0x1.62e42fefa39efp-1, ln2_lo = 0x1.abc9e3b39803fp-56;
  const double h = __builtin_fma(r, ln2, 1.0);
  double w = __builtin_fma(r, ln2_lo, __builtin_fma(r, ln2, 1.0 - h));
  w = __builtin_fma(r * r, p, w);
  w = __builtin_fma(ln2 * z_lo, h + w, w);
  return __builtin_ldexp(h + w, static_cast<int>(n));
}

// x^e, e > 0, for any x as pow returns it: 0, infinity and NaN stay, and a
// negative x has a power where e is a whole number (the fans of gamma = 5 / 3
// and 2 have such exponents) or x is infinite.
__device__ __forceinline__ double PowState(double x, double e) {
  const double a = rabs(x);
  const double r = (a > 0.0 && a <= 1.7976931348623157e308) ? PowPos(a, e) : a;
  if (__builtin_expect(!(x < 0.0), 1)) return r;
  if (__builtin_rint(e) == e) return __builtin_rint(0.5 * e) == 0.5 * e ? r : -r;
  return a <= 1.7976931348623157e308 ? __builtin_nan("") : r;
}

// x^e of the sampled star density (x a ratio of pressures).
template <bool MIXED> __device__ __forceinline__ double PowSample(double x, double e) {
  if constexpr (MIXED) {
    return static_cast<double>(__builtin_amdgcn_exp2f(
        static_cast<float>(e) * __builtin_amdgcn_logf(static_cast<float>(x))));
  } else {
    return PowState(x, e);
  }
}

template <int D, class T> __device__ __forceinline__ T SqNormScalar(const T* m) {
  if constexpr (D == 2) {
    return m[0] * m[0] + m[1] * m[1];
  } else {
    return (m[0] * m[0] + m[1] * m[1]) + m[2] * m[2];
  }
}

// PerfectGas::CompleteFromCons, scalar form (src/equations/PerfectGas.cpp:96-110).
template <int D>
__device__ __forceinline__ void CompleteFromConsScalar(double* q, const Gas<double>& g) {
  using I = Idx<D>;
  const double e_kin = 0.5 * SqNormScalar<D>(q + I::kMom) / q[I::kRho];
  const double e_int = q[I::kE] - e_kin;
  q[I::kP] = e_int / g.gm1inv;
  q[I::kA] = rsqrt_ieee(g.gamma * q[I::kP] / q[I::kRho]);
}

struct NewtonParams {
  double tol;      // 1e-7
  int max_it;      // 5000
};

struct MiddleState {
  double pM;
  double uM;
  int iterations;
  int converged;
  // At pM, per side: the shock's sqrt(A / (pM + B)) where pM is above the
  // side's pressure, else the rarefaction's (pM / p)^((gamma - 1) / (2 gamma)).
  double auxL;
  double auxR;
};

// Toro's pressure function of one side and its derivative, both at x (the
// Newton iteration needs the derivative at the point whose residual it just
// tested).  Shock branch: f = (x - p) r, r = sqrt(A / (x + B)) with 1 / A =
// (gamma + 1) rho / 2; the derivative r (1 - (x - p) / (2 (x + B))) takes
// 1 / (x + B) = r^2 / A.  Rarefaction branch: f = 2 a / (gamma - 1) (s - 1),
// s = (x/p)^((gamma-1)/(2 gamma)); the reference's second power,
// (x/p)^((gamma+1)/(-2 gamma)), is s / (x/p).
// The derivative only sets the Newton step, so its quotient and the step's are
// the refined reciprocal alone: a step is off by about 2^-48 of itself, which
// the next residual sees (the states' errors against 64-bit arithmetic did not
// grow).
struct SideFn {
  double p, y_p;   // pressure and its refined reciprocal
  double inv_A;    // (gamma + 1) rho / 2
  double B;        // (gamma - 1) / (gamma + 1) p
  double ra;       // rho a
  double c;        // 2 a / (gamma - 1)
  __device__ __forceinline__ double eval(double x, double exponent, double* df,
                                         double* aux) const {
    if (x > p) {
      const double r = NearArith::rsqrt((x + B) * inv_A);
      const double f = (x - p) * r;
      *aux = r;
      *df = r * __builtin_fma(-0.5 * f * inv_A, r, 1.0);
      return f;
    } else {
      const double t = NearArith::div(x, p, y_p);
      // t lies in [0, 1] or is NaN (no pressure on either side): 0 and NaN
      // are their own power, with an infinite or NaN slope
      const double s = t > 0.0 ? PowPos(t, exponent) : t;
      *aux = s;
      *df = t > 0.0 ? s * NearArith::inv(t * ra) : __builtin_huge_val() + t;
      return c * (s - 1.0);
    }
  }
};

// ComputeMiddleState with an explicit initial guess x0 (the reference's is
// 0.5 * (pL + pR)); uL, uR are the normal velocities.  The side functions at
// the final iterate, which the reference evaluates once more for the middle
// velocity, are the ones the last convergence test computed (same arguments,
// same values).
//
// The sides are taken by pressure (lo the lower): an iterate between the two
// pressures, where the mean and most star pressures lie, is a shock for lo
// and a rarefaction for hi in every lane, so a wave runs one branch a side;
// by left and right, half of its lanes take the other branch and the wave
// runs both.  The sums of the two sides do not depend on their order.
__device__ __forceinline__ MiddleState SolveMiddleState(double rhoL, double uL, double pL,
                                                        double aL, double rhoR, double uR,
                                                        double pR, double aR,
                                                        const Gas<double>& eq,
                                                        const NewtonParams& np, double x0) {
  const double g = eq.gamma;
  const double gp1 = g + 1.0;
  const double gm1 = g - 1.0;
  const double ratio = gm1 / gp1;
  const double y_gm1 = NearArith::inv(gm1);
  const double exponent = 0.5 * gm1 / g;
  auto side = [&](double rho, double p, double a) {
    SideFn s;
    s.p = p;
    s.y_p = NearArith::inv(p);
    s.inv_A = 0.5 * gp1 * rho;
    s.B = ratio * p;
    s.ra = rho * a;
    s.c = NearArith::div(2.0 * a, gm1, y_gm1);
    return s;
  };
  const bool swap = pR < pL;
  const SideFn lo = side(swap ? rhoR : rhoL, swap ? pR : pL, swap ? aR : aL);
  const SideFn hi = side(swap ? rhoL : rhoR, swap ? pL : pR, swap ? aL : aR);
  const double du = uR - uL;
  // NewtonIteration (NewtonIteration.hpp:28-52), one evaluation site.
  double x = x0;
  double d_lo, d_hi, aux_lo, aux_hi, f_lo, f_hi, fx;
  int counter = 0;
  while (true) {
    f_lo = lo.eval(x, exponent, &d_lo, &aux_lo);
    f_hi = hi.eval(x, exponent, &d_hi, &aux_hi);
    fx = f_lo + f_hi + du;
    if (!(rabs(fx) > np.tol && counter < np.max_it)) break;
    const double offset = fx * NearArith::inv(d_lo + d_hi);
    const double next = x - offset;
    x = ((next - next) != (next - next) || next < 0.0) ? 0.5 * x : next;
    counter += 1;
  }
  MiddleState ms;
  ms.pM = x;
  const double df = swap ? f_lo - f_hi : f_hi - f_lo;  // right less left
  ms.uM = 0.5 * (uL + uR) + 0.5 * df;
  ms.iterations = counter;
  ms.converged = !(counter == np.max_it && fx > np.tol);
  ms.auxL = swap ? aux_hi : aux_lo;
  ms.auxR = swap ? aux_lo : aux_hi;
  return ms;
}

template <int D, int DIR>
__device__ __forceinline__ MiddleState ComputeMiddleState(const double* L, const double* R,
                                                          const Gas<double>& eq,
                                                          const NewtonParams& np,
                                                          double x0) {
  using I = Idx<D>;
  return SolveMiddleState(L[I::kRho], L[I::kMom + DIR] / L[I::kRho], L[I::kP], L[I::kA],
                          R[I::kRho], R[I::kMom + DIR] / R[I::kRho], R[I::kP], R[I::kA], eq, np,
                          x0);
}

// Whether a speed of sound is one: positive and finite.
__device__ __forceinline__ bool IsGas(double a) { return __builtin_amdgcn_class(a, 0x180); }

// Normal velocities of a face's sides from their momenta; y: refined reciprocals
// of their densities.
__device__ __forceinline__ void FaceVelocities(double mL, double rhoL, double yL, double aL,
                                               double mR, double rhoR, double yR, double aR,
                                               double* uL, double* uR) {
  *uL = NearArith::div(mL, rhoL, yL);
  *uR = NearArith::div(mR, rhoR, yR);
  if (__builtin_expect(!(IsGas(aL) && IsGas(aR)), 0)) {
    *uL = NearArith::fix(*uL, mL, rhoL);
    *uR = NearArith::fix(*uR, mR, rhoR);
  }
}

// Largest signal speed of a face (ComputeSignals): uL less and uR plus the
// side's wave speed, a sqrt((gamma + 1) / (2 gamma) (pM / p - 1) + 1) for a
// shock, which is 1 / (rho r) with the side's r, and a for a rarefaction.
// The face's stable dt is dx / speed.
__device__ __forceinline__ double GodunovSpeed(double rhoL, double uL, double pL, double aL,
                                               double rhoR, double uR, double pR, double aR,
                                               const MiddleState& ms, double g, double* wL,
                                               double* wR) {
  *wL = ms.pM > pL ? NearArith::quot(1.0, rhoL * ms.auxL) : aL;
  *wR = ms.pM > pR ? NearArith::quot(1.0, rhoR * ms.auxR) : aR;
  if (__builtin_expect(!(IsGas(aL) && IsGas(aR)), 0)) {
    auto wave = [&](double p, double a) {
      return ms.pM > p ? a * rsqrt_ieee(((g + 1.0) * (ms.pM / p) + (g - 1.0)) / (2.0 * g)) : a;
    };
    *wL = wave(pL, aL);
    *wR = wave(pR, aR);
  }
  double s_max = 0.0;
  s_max = rmax(s_max, rabs(uL - *wL));
  s_max = rmax(s_max, rabs(uR + *wR));
  return s_max;
}

// SolveRiemannProblem: the complete state at x/t = 0 given the middle state
// (the cut cells' wall problems).
template <int D, int DIR>
__device__ __forceinline__ void SampleRiemann(double* state, const double* left,
                                              const double* right, double pM, double uM,
                                              const Gas<double>& eq) {
  using I = Idx<D>;
  constexpr int NQ = I::kComp;
  constexpr int M = I::kMom;
  auto set_momentum = [&](double momentum, const double* side) {
#pragma unroll
    for (int d = 0; d < D; ++d) state[M + d] = state[I::kRho] * (side[M + d] / side[I::kRho]);
    state[M + DIR] = momentum;
  };
  auto from_prim = [&]() {
    const double rhoE_kin = 0.5 * SqNormScalar<D>(state + M) / state[I::kRho];
    const double rhoE_internal = state[I::kP] * eq.gm1inv;
    state[I::kE] = rhoE_internal + rhoE_kin;
    state[I::kA] = rsqrt_ieee(eq.gamma * state[I::kP] / state[I::kRho]);
  };
  auto copy = [&](const double* s) {
#pragma unroll
    for (int k = 0; k < NQ; ++k) state[k] = s[k];
  };
  const double g = eq.gamma;
  const double gp1 = g + 1.0;
  const double gm1 = g - 1.0;
  if (0.0 <= uM) {
    const double uL = left[M + DIR] / left[I::kRho];
    const double aL = left[I::kA];
    const double pL = left[I::kP];
    const double p_ratio = pM / pL;
    const double g_ratio = gm1 / gp1;
    if (pM > pL) {
      const double shock_speed = uL - aL * rsqrt_ieee((gp1 * p_ratio + gm1) / (2.0 * g));
      if (shock_speed < 0.0) {
        state[I::kRho] = left[I::kRho] * (p_ratio + g_ratio) / (g_ratio * p_ratio + 1.0);
        set_momentum(state[I::kRho] * uM, left);
        state[I::kP] = pM;
        from_prim();
      } else {
        copy(left);
      }
    } else {
      const double aM = aL * PowState(p_ratio, gm1 / (2.0 * g));
      const double shock_speed_TL = uM - aM;
      const double shock_speed_HL = uL - aL;
      if (0.0 < shock_speed_HL) {
        copy(left);
      } else if (shock_speed_TL < 0.0) {
        state[I::kRho] = left[I::kRho] * PowState(p_ratio, 1.0 / g);
        set_momentum(state[I::kRho] * uM, left);
        state[I::kP] = pM;
        from_prim();
      } else {
        state[I::kRho] = left[I::kRho] * PowState(2.0 / gp1 + g_ratio * uL / aL, 2.0 / gm1);
        const double u = 2.0 / gp1 * (aL + 0.5 * gm1 * uL);
        set_momentum(state[I::kRho] * u, left);
        state[I::kP] = pL * PowState(2.0 / gp1 + g_ratio * uL / aL, 2.0 * g / gm1);
        from_prim();
      }
    }
  } else {
    const double uR = right[M + DIR] / right[I::kRho];
    const double aR = right[I::kA];
    const double pR = right[I::kP];
    const double p_ratio = pM / pR;
    const double g_ratio = gm1 / gp1;
    if (pM > pR) {
      const double shock_speed = uR + aR * rsqrt_ieee((gp1 * p_ratio + gm1) / (2.0 * g));
      if (0.0 < shock_speed) {
        state[I::kRho] = right[I::kRho] * (p_ratio + g_ratio) / (g_ratio * p_ratio + 1.0);
        set_momentum(state[I::kRho] * uM, right);
        state[I::kP] = pM;
        from_prim();
      } else {
        copy(right);
      }
    } else {
      const double aM = aR * PowState(p_ratio, gm1 / (2.0 * g));
      const double shock_speed_TR = uM + aM;
      const double shock_speed_HR = uR + aR;
      if (shock_speed_HR <= 0.0) {
        copy(right);
      } else if (shock_speed_TR >= 0.0) {
        state[I::kRho] = right[I::kRho] * PowState(p_ratio, 1.0 / g);
        set_momentum(state[I::kRho] * uM, right);
        state[I::kP] = pM;
        from_prim();
      } else {
        state[I::kRho] = right[I::kRho] * PowState(2.0 / gp1 - g_ratio * uR / aR, 2.0 / gm1);
        const double u = 2.0 / gp1 * (-aR + 0.5 * gm1 * uR);
        set_momentum(state[I::kRho] * u, right);
        state[I::kP] = pR * PowState(2.0 / gp1 - g_ratio * uR / aR, 2.0 * g / gm1);
        from_prim();
      }
    }
  }
}

// Godunov<PerfectGas<D>, ExactRiemannSolver> numeric flux between complete
// states L and R from their middle state (SolveRiemannProblem, then the
// physical flux of the state at x/t = 0).  y: refined reciprocals of the two
// densities; w: the sides' wave speeds (GodunovSpeed).  The side away from
// which the contact moves is mirrored onto the left, so both sides share one
// sequence of selects instead of two branch trees.
template <int D, int DIR, bool MIXED>
__device__ __forceinline__ void GodunovFlux(double* flux, const double* L, double yL,
                                            const double* R, double yR, const MiddleState& ms,
                                            double wL, double wR, const Gas<double>& eq) {
  using I = Idx<D>;
  constexpr int M = I::kMom;
  const double g = eq.gamma, gp1 = g + 1.0, gm1 = g - 1.0;
  const double g_ratio = gm1 / gp1;
  const bool left = 0.0 <= ms.uM;
  const double sign = left ? 1.0 : -1.0;
  double q[I::kComp];
#pragma unroll
  for (int k = 0; k < I::kComp; ++k) q[k] = left ? L[k] : R[k];
  const double y = left ? yL : yR;
  const double w = left ? wL : wR;
  const double aux = left ? ms.auxL : ms.auxR;
  const double rho = q[I::kRho], p = q[I::kP], a = q[I::kA];
  double vel[D];
#pragma unroll
  for (int d = 0; d < D; ++d) vel[d] = NearArith::div(q[M + d], rho, y);
  if (__builtin_expect(!IsGas(a), 0)) {
#pragma unroll
    for (int d = 0; d < D; ++d) vel[d] = NearArith::fix(vel[d], q[M + d], rho);
  }
  const double u = sign * vel[DIR];
  const double um = sign * ms.uM;
  const bool shock = ms.pM > p;
  // head of the wave left of x/t = 0: the side's own state (a head that stands
  // still counts for the right side only)
  const bool own = shock ? !(u - w < 0.0) : (left ? 0.0 < u - a : 0.0 <= u - a);
  const bool star = shock ? !own : (!own && um - a * aux < 0.0);
  const double t = NearArith::quot(ms.pM, p);
  double r0 = rho, p0 = p, u0 = u;
  if (star) {
    const double c = shock ? NearArith::quot(t + g_ratio, g_ratio * t + 1.0)
                           : PowSample<MIXED>(t, 1.0 / g);
    r0 = rho * c;
    p0 = ms.pM;
    u0 = um;
  } else if (!own) {
    const double b = 2.0 / gp1 + g_ratio * u / a;
    r0 = rho * PowState(b, 2.0 / gm1);
    p0 = p * PowState(b, 2.0 * g / gm1);
    u0 = 2.0 / gp1 * (a + 0.5 * gm1 * u);
  }
  vel[DIR] = own ? vel[DIR] : sign * u0;
  double mom[D], v2 = 0.0;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    mom[d] = own ? q[M + d] : r0 * vel[d];
    v2 += vel[d] * vel[d];
  }
  const double E = own ? q[I::kE] : p0 * eq.gm1inv + 0.5 * r0 * v2;
  flux[I::kRho] = mom[DIR];
#pragma unroll
  for (int d = 0; d < D; ++d) flux[M + d] = vel[DIR] * mom[d];
  flux[M + DIR] += p0;
  flux[I::kE] = vel[DIR] * (E + p0);
  if (!(0.0 < L[0] && 0.0 < R[0])) {  // no Riemann problem: the zero state's flux
    flux[I::kRho] = 0.0;
#pragma unroll
    for (int k = 1; k < D + 2; ++k) flux[k] = __builtin_nan("");
  }
}

} // namespace fvs
