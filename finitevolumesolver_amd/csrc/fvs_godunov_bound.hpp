// Certified speed bound of an exact-Godunov face, in single precision.
//
// The step-start CFL pass needs only the largest signal speed of a patch.
// A face whose speed provably stays below a known lower bound of it (the
// speed floor) needs no Newton solve; these bounds decide that without an
// iteration, from six floats a cell.  Single precision costs them nothing
// (every inequality is taken with a margin of 2^-18 or more, far above the
// rounding of a few float operations) and has one-instruction reciprocals and
// roots.  The pass issues more than 300 instructions a cell, so the test every
// face takes is the short one, and the tight one runs only in waves with a face
// that the short one leaves.
//
// Compiles for the host too, where tests/test_godunov_bound_f32.py holds it
// against the CPU oracle's signal speeds.
#pragma once

#include "fvs_physics.hpp"

namespace fvs {

// Newton iteration caps from which the pass skips faces at all, and from
// which it skips those of the wide class: from the mean pressure, Newton
// converges within 9 iterations (seen for gamma 5 / 3, 2 and 3; 6 up to 1.4) on
// pairs with pressure ratios up to 4 and |uR - uL| up to the smaller sound
// speed, and within 40 (21 seen) for ratios up to 1e6,
// parting speeds up to a quarter of what opens a vacuum and closing speeds up
// to 1e3 sound speeds (f is concave, so Newton climbs to a strong shock's
// pressure from below without overshooting); with a smaller cap the face is
// solved, so that the cap is reported where the reference throws.
constexpr int kGodunovFloorCap = 16;
constexpr int kGodunovWideCap = 64;

// A cell of the bound: 1 / rho, p, a^2 and the velocities.  A cell outside
// the ranges in which every product of the bounds stays representable
// (density and pressure within [1e-15, 1e15], sound speed up to 1e6), and one
// that is no gas, has a NaN pressure, which no test below passes.
template <int D> struct SpeedCell {
  float ir, p, a2;
  float u[D];
};

template <int D>
__device__ __forceinline__ SpeedCell<D> MakeSpeedCell(const double* q, const Gas<double>& g) {
  using FA = FastArith<double>;
  const FA::Inv ir = FA::inv(q[0]);
  SpeedCell<D> c;
  const double e_kin = FA::div(0.5 * SqNormArray<D>(q + 1), ir);
  const float p = static_cast<float>((q[D + 1] - e_kin) * g.gm1);
  c.ir = static_cast<float>(ir.y);
  c.a2 = static_cast<float>(g.gamma) * p * c.ir;
  const bool ok = c.ir >= 1e-15f && c.ir <= 1e15f && p >= 1e-15f && p <= 1e15f && c.a2 <= 1e12f;
  c.p = ok ? p : __builtin_nanf("");
#pragma unroll
  for (int d = 0; d < D; ++d) c.u[d] = static_cast<float>(FA::div(q[1 + d], ir));
  return c;
}

struct SpeedBound {
  float c;          // (gamma + 1) / 2
  float ratio;      // (gamma - 1) / (gamma + 1)
  float tol;        // Newton's residual
  float max_ratio;  // largest pressure ratio of the class
  bool wide;        // speeds below against aL^2 + aR^2, else the smaller a^2
  float part2;      // squared parting speed (uR > uL), at most
  float close2;     // squared closing speed, at most
  float du_max;     // |uR - uL| at which f still resolves tol
  float min_p_ir;   // least P / rho for which tol moves P by less than 2^-16
};

inline SpeedBound MakeSpeedBound(double gamma, double tol, int max_it) {
  SpeedBound b;
  const double c = 0.5 * (gamma + 1.0), ratio = (gamma - 1.0) / (gamma + 1.0);
  const bool wide = max_it >= kGodunovWideCap;
  b.c = static_cast<float>(c);
  b.ratio = static_cast<float>(ratio);
  b.tol = static_cast<float>(tol);
  b.max_ratio = wide ? 1e6f : 4.0f;
  b.wide = wide;
  const double part = 0.5 / (gamma - 1.0) < 1.25 ? 0.5 / (gamma - 1.0) : 1.25;
  b.part2 = wide ? static_cast<float>(part * part) : 1.0f;
  b.close2 = wide ? 1e6f : 1.0f;
  b.du_max = static_cast<float>(1e14 * tol);
  b.min_p_ir = static_cast<float>(tol * tol * 2.1 * (1.0 + ratio) * c * 0x1p32);
  return b;
}

// Both tests: whether a face's signal speeds max(|s0|, |s1|) stay below F.
//
// Toro's f(p) = fL(p) + fR(p) + (uR - uL) increases, so any P with f(P) >= 0
// bounds the star pressure.  At P >= max p both sides are on their shock
// branches (P - pK) rK(P), rK(P) = ((P + BK) cK)^(-1/2) with BK = ratio pK, cK
// = c rhoK.  Newton stops at |f| <= tol, which moves its result by at most
// tol over the slopes on [0, 2P], each at least rK(2P) / 2 >= 0.35 rK(P) (a
// rarefaction's slope is at least 1 / (rho a) = rK(pK)).  The speeds grow with
// the star pressure: |uK| + 1 / (rhoK rK(P)), the shock speed, bounds them (a
// rarefaction's aK is its value at pK <= P).
//
// Class: pressure ratio up to max_ratio, squared parting and closing speeds up
// to part2 and close2 times the smaller a^2 or (wide) aL^2 + aR^2, and speeds at
// which the rounding of f stays far below tol.
//
// Quick test, for every face of the pass: both rK are at least those of the
// larger density and B, so f(P) >= 2 (P - pmax) ((P + B) c rho)^(-1/2) + du,
// which is not negative from P = pmax + G + sqrt(G (pmax + B)) on, G = du^2 c
// rho / 4 (du the closing speed; none: P = pmax).
template <int D>
__device__ __forceinline__ bool QuickSpeedBelow(const SpeedCell<D>& L, float uL,
                                                const SpeedCell<D>& R, float uR,
                                                const SpeedBound& b, float F) {
  const float pmax = __builtin_fmaxf(L.p, R.p) + 0.0f * (L.p + R.p);  // NaN stays NaN
  const float pmin = __builtin_fminf(L.p, R.p);
  const float ir_max = __builtin_fmaxf(L.ir, R.ir), ir_min = __builtin_fminf(L.ir, R.ir);
  const float du = uR - uL;
  const float um = __builtin_fmaxf(__builtin_fabsf(uL), __builtin_fabsf(uR));
  const float dup = __builtin_fmaxf(-du, 0.0f) + um * 0x1p-20f;  // closing, rounded up
  const float k = 1.0f + b.ratio;
  const float G = dup * dup * (0.25f * b.c * (1.0f + 0x1p-16f)) * __builtin_amdgcn_rcpf(ir_min);
  const float P = (pmax + G + __builtin_amdgcn_sqrtf(G * k * pmax)) * (1.0f + 0x1p-15f);
  const float speed = (um + __builtin_amdgcn_sqrtf(P * (k * b.c) * ir_max)) * (1.0f + 0x1p-15f);
  return pmax <= b.max_ratio * pmin && du * du <= (du < 0.0f ? b.close2 : b.part2) *
                        (b.wide ? L.a2 + R.a2 : __builtin_fminf(L.a2, R.a2)) &&
         __builtin_fabsf(du) <= b.du_max &&
         P * ir_min >= b.min_p_ir && speed < F;
}

// Tight test, for the faces that the quick one leaves: P = max p serves when
// the lower side's branch covers the closing speed, else max p plus twice the
// missing speed over the slopes, with f(P) >= 0 verified.
template <int D>
__device__ __forceinline__ bool SpeedBelow(const SpeedCell<D>& L, float uL,
                                           const SpeedCell<D>& R, float uR, const SpeedBound& b,
                                           float F) {
  constexpr float kUp = 1.0f + 0x1p-18f, kDn = 1.0f - 0x1p-18f;
  const bool swap = R.p < L.p;
  const float pmin = swap ? R.p : L.p, pmax = swap ? L.p : R.p;
  const float ir_lo = swap ? R.ir : L.ir, ir_hi = swap ? L.ir : R.ir;
  const float u_lo = swap ? uR : uL, u_hi = swap ? uL : uR;
  const float du = uR - uL;
  const float span = __builtin_fabsf(uL) + __builtin_fabsf(uR);
  const bool in_class = pmin > 0.0f && pmax <= b.max_ratio * pmin &&
                        du * du <= (du < 0.0f ? b.close2 : b.part2) *
                        (b.wide ? L.a2 + R.a2 : __builtin_fminf(L.a2, R.a2)) &&
         __builtin_fabsf(du) <= b.du_max;
  const float need = span * 0x1p-20f - du;  // closing speed, rounded up
  const float c_lo = b.c * __builtin_amdgcn_rcpf(ir_lo), c_hi = b.c * __builtin_amdgcn_rcpf(ir_hi);
  const float B_lo = b.ratio * pmin, B_hi = b.ratio * pmax;
  const float p_lo = pmin * (1.0f + 0x1p-22f), p_hi = pmax * (1.0f + 0x1p-22f);
  float r_lo = __builtin_amdgcn_rsqf((pmax + B_lo) * c_lo);
  float r_hi = __builtin_amdgcn_rsqf((pmax + B_hi) * c_hi);
  const float f0 = (pmax * (1.0f - 0x1p-22f) - p_lo) * r_lo * kDn;
  float P = p_hi;
  bool covered = f0 >= need;
  if (!covered) {
    P = (pmax + 2.0f * (need - f0) * __builtin_amdgcn_rcpf(r_lo + r_hi)) * kUp;
    r_lo = __builtin_amdgcn_rsqf((P + B_lo) * c_lo);
    r_hi = __builtin_amdgcn_rsqf((P + B_hi) * c_hi);
    covered = ((P - p_lo) * r_lo + (P - p_hi) * r_hi) * kDn >= need;
  }
  const float Peff = P + b.tol * __builtin_amdgcn_rcpf(0.35f * (r_lo + r_hi) * kDn);
  const float s_lo = __builtin_amdgcn_sqrtf((Peff + B_lo) * b.c * ir_lo);
  const float s_hi = __builtin_amdgcn_sqrtf((Peff + B_hi) * b.c * ir_hi);
  const float speed =
      __builtin_fmaxf(__builtin_fabsf(u_lo) + s_lo, __builtin_fabsf(u_hi) + s_hi) * kUp;
  return in_class && covered && Peff <= 2.0f * P && speed < F;
}

}  // namespace fvs
