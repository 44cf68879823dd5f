// HLLEM face speeds from per-cell ingredients, shared by the fused sweeps and
// CFL passes, and the lane shifts of what they pass between lanes.
#pragma once

#include "fvs_lanes.hpp"
#include "fvs_physics.hpp"

namespace fvs {

// Largest of two signal speeds; a NaN speed never wins (as a NaN face dt
// never wins the minimum).
__device__ __forceinline__ double SMax(double a, double b) { return __builtin_fmax(a, b); }

__device__ __forceinline__ double WaveMaxSpeed(double s) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s = SMax(s, __shfl_xor(s, off, 64));
  return s;
}

// Per-cell ingredients of Hllem::ComputeStableDt
// (src/equations/perfect_gas/HllemMethod.hpp:1152-1216): sqrt(rho), the
// velocity, the enthalpy (E + p) / rho and the speed of sound.  A face's dt
// combines two of them with exactly the reference's operations.
template <int D> struct DtCell {
  double sq;
  double u[D];
  double h;
  double a;
};

template <int D, class A>
__device__ __forceinline__ DtCell<D> MakeDtCell(const double* u, const Gas<double>& g) {
  double q[D + 4];
#pragma unroll
  for (int c = 0; c < D + 2; ++c) q[c] = u[c];
  const typename A::Inv ir = CompleteFromCons<D, double, A>(q, g);
  DtCell<D> r;
  r.sq = A::sqrt(q[0]);
#pragma unroll
  for (int i = 0; i < D; ++i) r.u[i] = A::div(q[1 + i], ir);
  r.h = A::div(q[D + 1] + q[D + 2], ir);
  r.a = q[D + 3];
  return r;
}

// The face's largest signal speed max(|sL|, |sR|); its stable dt is
// dx / speed (reduced per block by BlockSpeedToPartials).
template <int D, int DIR, class A>
__device__ __forceinline__ double FaceSpeed(const DtCell<D>& L, const DtCell<D>& R,
                                            double gm1) {
  const double sqRhoSum = L.sq + R.sq;
  const typename A::Inv isum = A::inv(sqRhoSum);
  const double wL = A::div(L.sq, isum);
  const double wR = A::div(R.sq, isum);
  double roeU[D];
#pragma unroll
  for (int i = 0; i < D; ++i) roeU[i] = wL * L.u[i] + wR * R.u[i];
  const double roeH = wL * L.h + wR * R.h;
  double sq = roeU[0] * roeU[0];
#pragma unroll
  for (int i = 1; i < D; ++i) sq += roeU[i] * roeU[i];
  const double roeA2 = gm1 * (roeH - 0.5 * sq);
  const double roeA = A::sqrt(roeA2);
  const double maxA = A::max(L.a, R.a);
  const double sL = A::min(L.u[DIR] - maxA, roeU[DIR] - roeA);
  const double sR = A::max(roeU[DIR] + roeA, R.u[DIR] + maxA);
  return A::max(rabs(sL), rabs(sR));
}

template <int D>
__device__ __forceinline__ BoundCell<D> ShflUp(const BoundCell<D>& v) {
  BoundCell<D> r;
#pragma unroll
  for (int i = 0; i < D; ++i) r.u[i] = ShiftUp(v.u[i]);
  r.a2 = ShiftUp(v.a2);
  return r;
}

template <int D>
__device__ __forceinline__ DtCell<D> ShflUp(const DtCell<D>& v) {
  DtCell<D> r;
  r.sq = ShiftUp(v.sq);
#pragma unroll
  for (int i = 0; i < D; ++i) r.u[i] = ShiftUp(v.u[i]);
  r.h = ShiftUp(v.h);
  r.a = ShiftUp(v.a);
  return r;
}

} // namespace fvs
