// Exact-Godunov flux method on gfx950: FluxMethod<Godunov<PerfectGas<D>,
// ExactRiemannSolver>> (include/fub/flux_method/GodunovMethod.hpp:130-199).
//
// Fused first-order sweeps (X: slot-mapped lanes like the HLLEM sweep; Y/Z:
// pencil march).  The face flux and the face's CFL signal speeds need the
// same Riemann problem of the same two cell states, so one FP64 Newton
// iteration serves both (the reference solves it twice: once in
// ComputeNumericFlux, once in ComputeSignals).  An optional per-face initial
// guess (the learned star pressure) replaces 0.5 (pL + pR); Newton itself,
// its tolerance and its safeguards are unchanged.  Newton statistics
// (iterations, non-converged faces) are accumulated per workgroup.
#include "fvs_godunov_bound.hpp"
#include "fvs_internal.hpp"
#include "fvs_lanes.hpp"
#include "fvs_mlp_infer.hpp"
#include "fvs_riemann.hpp"
#include "fvs_views.hpp"
#include "fvs_xslots.hpp"

#include <cstring>
#include <type_traits>

namespace fvs {

namespace {

constexpr int kBlock = 256;
constexpr unsigned long long kInfKey = 0x7ff0000000000000ull;

__device__ __forceinline__ int64_t Clamp(int64_t i, int64_t n) {
  return i < 0 ? 0 : (i >= n ? n - 1 : i);
}
__device__ __forceinline__ unsigned long long KMin(unsigned long long a, unsigned long long b) {
  return b < a ? b : a;
}
__device__ __forceinline__ unsigned long long WaveMinKey(unsigned long long k) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) k = KMin(k, __shfl_xor(k, off, 64));
  return k;
}
__device__ __forceinline__ unsigned long long WaveSum(unsigned long long k) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) k += __shfl_xor(k, off, 64);
  return k;
}
__device__ __forceinline__ unsigned long long WaveMaxU(unsigned long long k) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(k, off, 64);
    k = o > k ? o : k;
  }
  return k;
}

// Key of the stable dt dx / speed of a largest signal speed (+inf for 0): a
// rounded quotient falls monotonically with its denominator, so the smallest
// face dt is the quotient by the largest speed.
__device__ __forceinline__ unsigned long long SpeedKey(double dx, double speed) {
  return speed > 0.0 ? DtKey(DivRn(dx, speed)) : kInfKey;
}

// Block reduction of (largest speed, sum iterations, max iterations,
// non-converged faces, faces) to partials[block * 5 + i], the speed as the
// key of its stable dt.
template <int WAVES>
__device__ void BlockReduceGodunov(double speed, double dx, unsigned long long iters,
                                   unsigned long long maxit, unsigned long long fails,
                                   unsigned long long faces, unsigned long long* out) {
  __shared__ unsigned long long s[5][WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned long long key = WaveMinKey(SpeedKey(dx, speed));
  iters = WaveSum(iters);
  maxit = WaveMaxU(maxit);
  fails = WaveSum(fails);
  faces = WaveSum(faces);
  if (lane == 0) {
    s[0][wave] = key;
    s[1][wave] = iters;
    s[2][wave] = maxit;
    s[3][wave] = fails;
    s[4][wave] = faces;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long r[5] = {s[0][0], s[1][0], s[2][0], s[3][0], s[4][0]};
    for (int w = 1; w < WAVES; ++w) {
      r[0] = KMin(r[0], s[0][w]);
      r[1] += s[1][w];
      r[2] = s[2][w] > r[2] ? s[2][w] : r[2];
      r[3] += s[3][w];
      r[4] += s[4][w];
    }
    for (int i = 0; i < 5; ++i) out[i] = r[i];
  }
  __syncthreads();
}

struct GodunovArgs {
  const double* in[5];
  double* out[5];
  int64_t n[3];
  double dx;
  const double* dt_ptr;
  double dt_val;
  double gamma;
  double gm1inv;
  double tol;
  int max_it;
  const double* guess;   // per-face initial guess (nullable)
  const short* tiles;    // learned guess computed inline (nullable)
  const float* bias;
  unsigned long long* partials;  // 5 per workgroup
  int* halt;
  int seg;
  int update;            // 0: only fluxes' Newton + CFL (no state write)
  int limiter;           // MUSCL-Hancock sweeps
  int check;             // MUSCL-Hancock: the cells' CFL check against dt
  SpeedBound bound;
};

__device__ __forceinline__ Gas<double> GasOf(const GodunovArgs& a) {
  Gas<double> g;
  g.gamma = a.gamma;
  g.gm1inv = a.gm1inv;
  g.gm1 = a.gamma - 1.0;
  return g;
}

// A complete state in registers with the refined reciprocal of its density.
template <int D> struct CellState {
  double q[D + 4];
  double y;
};

// Newton from a caller's seed (learned or given), with the reference's
// initial guess, the mean pressure, as the fallback.  A seed that is not a
// finite positive pressure (an overflowed or underflowed network output) is
// not tried; a run from the seed that does not converge, or ends on a
// pressure that is not finite and non-negative, is redone from the mean.
// Both count as a fallback.
template <int D>
__device__ __forceinline__ MiddleState SeededMiddleState(const CellState<D>& L, double uL,
                                                         const CellState<D>& R, double uR,
                                                         const Gas<double>& g,
                                                         const NewtonParams& np, bool seeded,
                                                         double seed, double mean, int* iters,
                                                         int* fallback) {
  using I = Idx<D>;
  const bool usable = seeded && seed > 0.0 && seed <= 1.7976931348623157e308;
  double x0 = usable ? seed : mean;
  int it = 0, fb = seeded && !usable;
  MiddleState ms;
  while (true) {  // one Newton site for the seed and the mean
    ms = SolveMiddleState(L.q[0], uL, L.q[I::kP], L.q[I::kA], R.q[0], uR, R.q[I::kP], R.q[I::kA],
                          g, np, x0);
    it += ms.iterations;
    if (!usable || fb || (ms.converged && ms.pM >= 0.0 && ms.pM <= 1.7976931348623157e308)) break;
    x0 = mean;
    fb = 1;
  }
  *iters = it;
  *fallback = fb;
  return ms;
}

// Largest signal speed of the face between complete states L and R (normal
// momenta mL, mR), from Newton; acc (nullable): iterations, their maximum,
// solves that hit the cap.
template <int D>
__device__ __forceinline__ double CellFaceSpeed(const double* L, double mL, const double* R,
                                                double mR, const Gas<double>& g, double tol,
                                                int max_it, unsigned long long* acc) {
  using I = Idx<D>;
  double uL, uR;
  FaceVelocities(mL, L[0], NearArith::inv(L[0]), L[I::kA], mR, R[0], NearArith::inv(R[0]),
                 R[I::kA], &uL, &uR);
  NewtonParams np;
  np.tol = tol;
  np.max_it = max_it;
  const MiddleState ms = SolveMiddleState(L[0], uL, L[I::kP], L[I::kA], R[0], uR, R[I::kP],
                                          R[I::kA], g, np, 0.5 * (L[I::kP] + R[I::kP]));
  if (acc) {
    const unsigned long long it = static_cast<unsigned long long>(ms.iterations);
    acc[0] += it;
    acc[1] = it > acc[1] ? it : acc[1];
    acc[2] += ms.converged ? 0 : 1;
  }
  double wL, wR;
  return GodunovSpeed(L[0], uL, L[I::kP], L[I::kA], R[0], uR, R[I::kP], R[I::kA], ms, g.gamma, &wL,
                      &wR);
}

// A quotient by NearArith, with special results where FIX.
template <bool FIX> __device__ __forceinline__ double Quot(double a, double b, double y) {
  const double q = NearArith::div(a, b, y);
  return FIX ? NearArith::fix(q, a, b) : q;
}

// Pressure and speed of sound of a conservative state; SCALAR: kinetic energy
// in the order of the scalar path (fvs_riemann.hpp).  y_g = inv(gm1inv).  A
// state that is no gas (IsGas) is completed with FIX.
template <int D, bool SCALAR, bool FIX>
__device__ __forceinline__ void CompleteNear(CellState<D>& c, const Gas<double>& g, double y_g) {
  using I = Idx<D>;
  c.y = NearArith::inv(c.q[0]);
  const double sq = SCALAR ? SqNormScalar<D>(c.q + 1) : SqNormArray<D>(c.q + 1);
  const double e_int = c.q[I::kE] - Quot<FIX>(0.5 * sq, c.q[0], c.y);
  c.q[I::kP] = Quot<FIX>(e_int, g.gm1inv, y_g);
  c.q[I::kA] = NearArith::sqrt(Quot<FIX>(g.gamma * c.q[I::kP], c.q[0], c.y));
}

// A first-order cell.
template <int D>
__device__ __forceinline__ void Complete(CellState<D>& c, const Gas<double>& g, double y_g) {
  CompleteNear<D, false, false>(c, g, y_g);
  if (__builtin_expect(!IsGas(c.q[Idx<D>::kA]), 0)) CompleteNear<D, false, true>(c, g, y_g);
}

// MUSCL-Hancock half-step states of one cell at its left and right face
// (MusclHancockMethod.hpp:419-485) in the sequential driver's arithmetic.
template <int D, int DIR, int LIM, bool FIX>
__device__ __forceinline__ void HalfStep(const double* um, const double* u0, const double* up,
                                          double lh, const Gas<double>& g, double y_g,
                                          CellState<D>& recL, CellState<D>& recR) {
  using I = Idx<D>;
  constexpr int NC = D + 2;
  double f[2][NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const double s = LimitedSlope<LIM>(um[k], u0[k], up[k]);
    recL.q[k] = u0[k] - 0.5 * s;
    recR.q[k] = u0[k] + 0.5 * s;
  }
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const double* q = side == 0 ? recL.q : recR.q;
    const double y = NearArith::inv(q[0]);
    const double e_kin = Quot<FIX>(0.5 * SqNormScalar<D>(q + 1), q[0], y);
    const double p = Quot<FIX>(q[I::kE] - e_kin, g.gm1inv, y_g);
    const double v = Quot<FIX>(q[1 + DIR], q[0], y);
    f[side][0] = q[1 + DIR];
#pragma unroll
    for (int d = 0; d < D; ++d) f[side][1 + d] = v * q[1 + d];
    f[side][1 + DIR] += p;
    f[side][I::kE] = v * (q[I::kE] + p);
  }
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const double dq = lh * (f[0][k] - f[1][k]);
    recR.q[k] += dq;
    recL.q[k] += dq;
  }
  CompleteNear<D, true, FIX>(recR, g, y_g);
  CompleteNear<D, true, FIX>(recL, g, y_g);
}

// Which states of a cell a caller reads.
constexpr int kLeftState = 1, kRightState = 2, kBothStates = 3;

// Any cell.  A special quotient of one state's flux makes neither state a gas,
// so the states that are read tell (the other one's are never computed).
template <int D, int DIR, int LIM, int USE>
__device__ __forceinline__ void Recon(const double* um, const double* u0, const double* up,
                                      double lh, const Gas<double>& g, double y_g,
                                      CellState<D>& recL, CellState<D>& recR) {
  using I = Idx<D>;
  HalfStep<D, DIR, LIM, false>(um, u0, up, lh, g, y_g, recL, recR);
  const bool gas = (!(USE & kLeftState) || IsGas(recL.q[I::kA])) &&
                   (!(USE & kRightState) || IsGas(recR.q[I::kA]));
  if (__builtin_expect(!gas, 0))
    HalfStep<D, DIR, LIM, true>(um, u0, up, lh, g, y_g, recL, recR);
}

template <int D, int DIR, int USE = kBothStates>
__device__ __forceinline__ void ReconAny(int limiter, const double* um, const double* u0,
                                         const double* up, double lh, const Gas<double>& g,
                                         double y_g, CellState<D>& recL, CellState<D>& recR) {
  switch (limiter) {
  case kMinMod: Recon<D, DIR, kMinMod, USE>(um, u0, up, lh, g, y_g, recL, recR); break;
  case kVanLeer: Recon<D, DIR, kVanLeer, USE>(um, u0, up, lh, g, y_g, recL, recR); break;
  case kNoLimiter: Recon<D, DIR, kNoLimiter, USE>(um, u0, up, lh, g, y_g, recL, recR); break;
  default: Recon<D, DIR, kNoGradient, USE>(um, u0, up, lh, g, y_g, recL, recR); break;
  }
}

// Per-thread sums of a sweep: largest signal speed, Newton iterations (sum
// and maximum), faces that hit the cap, faces and (high bits) fallbacks.
struct FaceSums {
  double smax = 0.0;
  unsigned iters = 0, max_it = 0, fails = 0, faces = 0, fallbacks = 0;
  __device__ __forceinline__ unsigned long long packed_faces() const {
    return faces + (static_cast<unsigned long long>(fallbacks) << 32);
  }
};

// One face: Newton (shared by flux and CFL), flux and, from the same middle
// state, the largest signal speed of a first-order face.  MIXED: the sampled
// star density's power in single precision.
template <int D, int DIR, bool MIXED>
__device__ __forceinline__ void GodunovFace(const CellState<D>& L, const CellState<D>& R,
                                            double guess, bool has_guess, const GodunovArgs& a,
                                            const Gas<double>& g, double* F, bool count,
                                            bool speeds, FaceSums& sums) {
  using I = Idx<D>;
  NewtonParams np;
  np.tol = a.tol;
  np.max_it = a.max_it;
  double uL, uR;
  FaceVelocities(L.q[1 + DIR], L.q[0], L.y, L.q[I::kA], R.q[1 + DIR], R.q[0], R.y, R.q[I::kA], &uL,
                 &uR);
  const double mean = 0.5 * (L.q[I::kP] + R.q[I::kP]);
  int it, fallback;
  const MiddleState ms = SeededMiddleState<D>(L, uL, R, uR, g, np, has_guess, guess, mean, &it,
                                              &fallback);
  double wL, wR;
  const double speed = GodunovSpeed(L.q[0], uL, L.q[I::kP], L.q[I::kA], R.q[0], uR, R.q[I::kP],
                                    R.q[I::kA], ms, g.gamma, &wL, &wR);
  GodunovFlux<D, DIR, MIXED>(F, L.q, L.y, R.q, R.y, ms, wL, wR, g);
  if (count) {
    const unsigned n = static_cast<unsigned>(it);
    sums.iters += n;
    sums.max_it = n > sums.max_it ? n : sums.max_it;
    sums.fails += ms.converged ? 0 : 1;
    sums.faces += 1;
    sums.fallbacks += fallback;
    if (speeds) sums.smax = __builtin_fmax(sums.smax, speed);
  }
}

// CFL check of a MUSCL-Hancock sweep's face, whose signal speeds are those of
// the two cells and not of the half-step states the flux solves: the check
// only decides pass or fail, so a face certified to stay below dx / dt
// (`crit`, less a margin) needs no solve; the others are solved, and the
// reported minimum is exact wherever the check fails.  Called by the whole
// wave.
template <int D, int DIR>
__device__ __forceinline__ void CheckFace(const double* uL, const double* uR, bool face,
                                          const GodunovArgs& a, const Gas<double>& g, float crit,
                                          FaceSums& sums) {
  const SpeedCell<D> l = MakeSpeedCell<D>(uL, g), r = MakeSpeedCell<D>(uR, g);
  bool pass = !face || QuickSpeedBelow<D>(l, l.u[DIR], r, r.u[DIR], a.bound, crit);
  if (__builtin_expect(__any(!pass), 0)) {
    pass = !face || SpeedBelow<D>(l, l.u[DIR], r, r.u[DIR], a.bound, crit);
    if (!pass) {
      double L[D + 4], R[D + 4];
#pragma unroll
      for (int k = 0; k < D + 2; ++k) {
        L[k] = uL[k];
        R[k] = uR[k];
      }
      CompleteFromCons<D>(L, g);
      CompleteFromCons<D>(R, g);
      sums.smax = __builtin_fmax(sums.smax, CellFaceSpeed<D>(L, L[1 + DIR], R, R[1 + DIR], g,
                                                             a.tol, a.max_it, nullptr));
    }
  }
}

// X sweep: the slot walk of the HLLEM X sweep (fvs_xslots.hpp): persistent
// waves over 64-slot chunks of the rows' cells and ghosts, neighbours by DPP,
// the next chunk's load in flight behind Newton.  LEARNED: the network's guess
// is inferred inline (a.tiles set); without it the kernel carries none of the
// matrix-core code or its registers.  MUSCL: half-step states (FP64, mean
// guess) and, with a.check, the cells' CFL check; a ghost slot's slopes vanish
// (its clamped value equals its inner neighbour's; NoLimiter's outer neighbour
// is replaced).  Bound by Newton's FP64 instructions (1560 a cell at 256^3,
// smooth and strong waves; VALU busy 76%) at two waves per SIMD (180 to 250
// registers; held to 168 or 128 it spills and runs 1.5 to 3 times slower).
// 384^3 strong-wave blocks, faces seeded by the CFL pass: 3.9 -> 2.9 ms a sweep
// against one wave per 62 slots with LDS shuffles (3.9 ms from the mean guess,
// as now); MUSCL over 256^3: 8.6 -> 2.8 ms a step against the patch operators'
// passes (fluxes, stable dt, update, completion).
// LONG: rows of kXLongRow cells or more, whose offsets take 64 bits.
template <int D, bool MIXED, bool LEARNED, bool MUSCL, bool LONG>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void GodunovSweepX(GodunovArgs a) {
  constexpr int NC = D + 2, NQ = D + 4;
  if (a.halt && *a.halt) return;
  const int64_t nx = a.n[0];
  const uint32_t Q = static_cast<uint32_t>(a.n[1] * a.n[2]) * static_cast<uint32_t>(nx + 2);
  const int64_t nchunks = (static_cast<int64_t>(Q) + kXOwned - 1) / kXOwned;
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = static_cast<int64_t>(gridDim.x) * (kBlock / 64);
  const bool owned = lane >= 2 && lane < 2 + kXOwned;
  const Gas<double> g = GasOf(a);
  const double y_g = NearArith::inv(g.gm1inv);
  const double dt = a.dt_ptr ? *a.dt_ptr : a.dt_val;
  const double dt_dx = DivRn(dt, a.dx);
  const double lh = DivRn(0.5 * dt, a.dx);
  const float crit = static_cast<float>((a.dx / dt) * (1.0 - 0x1p-20));
  XSlotWalker walk(nx, Q, nwaves, lane);
  auto locate = [&](int64_t c) {
    bool valid;
    uint32_t row, sl;
    walk.RowSlot(c, &valid, &row, &sl);
    return walk.Make(valid, row, sl, __builtin_amdgcn_readfirstlane(row));
  };
  auto load = [&](const XSlot& s, double* u) {
    if constexpr (LONG) {
#pragma unroll
      for (int k = 0; k < NC; ++k) u[k] = a.in[k][s.wbase + s.rbase + Clamp(s.cell, nx)];
    } else {
      const uint32_t off = 8u * (s.rbase + static_cast<uint32_t>(Clamp(s.cell, nx)));
#pragma unroll
      for (int k = 0; k < NC; ++k)
        u[k] = *reinterpret_cast<const double*>(
            reinterpret_cast<const char*>(a.in[k] + s.wbase) + off);
    }
  };
  FaceSums sums;
  int64_t c = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) +
              __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  walk.Place(c < nchunks ? c : 0);
  XSlot cur = locate(c < nchunks ? c : 0);
  double u[NC];
  if (c < nchunks) load(cur, u);
  for (; c < nchunks; c += nwaves) {
    const int64_t cn = c + nwaves;
    walk.Next<LONG>(c, cn, nchunks);
    const XSlot nxt = locate(cn < nchunks ? cn : c);
    double un[NC];
    if (cn < nchunks) load(nxt, un);
    const bool real = cur.valid && cur.cell >= 0 && cur.cell < nx;
    const bool face_lane = cur.valid && lane >= 2 && lane <= 2 + kXOwned && cur.sl >= 1;
    CellState<D> L, R;  // states left and right of the slot's lower face
    double ul[NC];
    if constexpr (MUSCL) {
      double up[NC];
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        ul[k] = ShiftUp(u[k]);
        up[k] = ShiftDown(u[k]);
      }
      double um[NC];
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        um[k] = (a.limiter == kNoLimiter && cur.cell < 0) ? u[k] : ul[k];
        if (a.limiter == kNoLimiter && cur.cell >= nx) up[k] = u[k];
      }
      ReconAny<D, 0>(a.limiter, um, u, up, lh, g, y_g, R, L);
    } else {
#pragma unroll
      for (int k = 0; k < NC; ++k) R.q[k] = u[k];
      Complete<D>(R, g, y_g);
      L = R;
    }
#pragma unroll
    for (int k = 0; k < NQ; ++k) L.q[k] = ShiftUp(L.q[k]);
    L.y = ShiftUp(L.y);
    double guess = 0.0;
    if constexpr (LEARNED) {
      // every lane takes part in the wave's matrix-core step
      guess = mlp::LearnedGuess<D, 0>(L.q, R.q, a.tiles, a.bias);
    }
    double F[NC];
    if (face_lane) {
      if constexpr (!LEARNED && !MUSCL) {
        if (a.guess) {
          const int64_t row = (cur.wbase + cur.rbase) / nx;
          guess = a.guess[row * (nx + 1) + static_cast<int64_t>(cur.sl) - 1];
        }
      }
      GodunovFace<D, 0, MIXED>(L, R, guess, LEARNED || a.guess != nullptr, a, g, F, owned, !MUSCL,
                               sums);
    } else {
#pragma unroll
      for (int k = 0; k < NC; ++k) F[k] = 0.0;
    }
    double Fnext[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) Fnext[k] = ShiftDown(F[k]);
    if (a.update && owned && real) {
      if constexpr (LONG) {
#pragma unroll
        for (int k = 0; k < NC; ++k)
          a.out[k][cur.wbase + cur.rbase + cur.cell] = u[k] + dt_dx * (F[k] - Fnext[k]);
      } else {
        const uint32_t off = 8u * (cur.rbase + static_cast<uint32_t>(cur.cell));
#pragma unroll
        for (int k = 0; k < NC; ++k)
          *reinterpret_cast<double*>(reinterpret_cast<char*>(a.out[k] + cur.wbase) + off) =
              u[k] + dt_dx * (F[k] - Fnext[k]);
      }
    }
    if constexpr (MUSCL) {
      if (a.check) CheckFace<D, 0>(ul, u, owned && face_lane, a, g, crit, sums);
    }
    cur = nxt;
#pragma unroll
    for (int k = 0; k < NC; ++k) u[k] = un[k];
  }
  BlockReduceGodunov<kBlock / 64>(sums.smax, a.dx, sums.iters, sums.max_it, sums.fails, sums.packed_faces(),
                                  a.partials + 5 * blockIdx.x);
}

// Y / Z sweep: one thread per pencil marching a segment with the cell before
// (and, MUSCL, around) the face in registers and the next cell's load in
// flight.  Bound by Newton's FP64 instructions, like the X sweep (1080 a cell,
// VALU busy 74%).
template <int D, int DIR, bool MIXED, bool LEARNED, bool MUSCL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void GodunovSweepPencil(GodunovArgs a) {
  constexpr int NC = D + 2;
  if (a.halt && *a.halt) return;
  const int64_t nx = a.n[0], ny = a.n[1];
  const int64_t nd = a.n[DIR];
  const int64_t npencil = (DIR == 1) ? nx * a.n[2] : nx * ny;
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  const bool active = p0 < npencil;
  // Lanes past the last pencil repeat it (all lanes of a wave march together,
  // which the inline matrix-core guess needs); their results are not kept.
  const int64_t p = active ? p0 : npencil - 1;
  const int64_t stride = (DIR == 1) ? nx : nx * ny;
  const int64_t base = (DIR == 1) ? (p % nx) + (p / nx) * nx * ny : p;
  // Face (x, j, z) of direction DIR in the face box (n with n[DIR] + 1).
  const int64_t fbase = (DIR == 1) ? (p % nx) + (p / nx) * nx * (ny + 1) : p;
  const int64_t j0 = static_cast<int64_t>(blockIdx.y) * a.seg;
  const int64_t j1 = (j0 + a.seg < nd) ? j0 + a.seg : nd;
  const Gas<double> g = GasOf(a);
  const double y_g = NearArith::inv(g.gm1inv);
  const double dt = a.dt_ptr ? *a.dt_ptr : a.dt_val;
  const double dt_dx = DivRn(dt, a.dx);
  const double lh = DivRn(0.5 * dt, a.dx);
  const float crit = static_cast<float>((a.dx / dt) * (1.0 - 0x1p-20));

  FaceSums sums;
  auto load = [&](double* u, int64_t j) {
    const int64_t off = base + Clamp(j, nd) * stride;
#pragma unroll
    for (int k = 0; k < NC; ++k) u[k] = a.in[k][off];
  };
  double Um[NC], U0[NC], Unext[NC], Fprev[NC];
  load(Um, j0 - 1);
  load(U0, j0);
  load(Unext, j0 + 1);
  CellState<D> L;
  if constexpr (MUSCL) {
    // Half-step state of cell j0 - 1 (a ghost at j0 = 0, whose clamped
    // neighbours give it no slope).
    double Umm[NC];
    load(Umm, j0 - 2);
    CellState<D> unused;
    if (j0 == 0)
      Recon<D, DIR, kNoGradient, kRightState>(Um, Um, Um, lh, g, y_g, unused, L);
    else
      ReconAny<D, DIR, kRightState>(a.limiter, Umm, Um, U0, lh, g, y_g, unused, L);
  } else {
#pragma unroll
    for (int k = 0; k < NC; ++k) L.q[k] = Um[k];
    Complete<D>(L, g, y_g);
  }
  for (int64_t j = j0; j <= j1; ++j) {
    double Up[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) Up[k] = Unext[k];
    if (j + 1 < nd && j < j1) load(Unext, j + 2);
    CellState<D> R, Lnext;
    if constexpr (MUSCL) {
      if (j < nd)
        ReconAny<D, DIR>(a.limiter, Um, U0, Up, lh, g, y_g, R, Lnext);
      else
        Recon<D, DIR, kNoGradient, kLeftState>(U0, U0, U0, lh, g, y_g, R, Lnext);
    } else {
#pragma unroll
      for (int k = 0; k < NC; ++k) R.q[k] = U0[k];
      Complete<D>(R, g, y_g);
      Lnext = R;
    }
    double F[NC];
    double guess = 0.0;
    if constexpr (LEARNED) {
      guess = mlp::LearnedGuess<D, DIR>(L.q, R.q, a.tiles, a.bias);
    } else if constexpr (!MUSCL) {
      if (a.guess) guess = a.guess[fbase + j * stride];
    }
    const bool mine = active && (j < j1 || j1 == nd);
    GodunovFace<D, DIR, MIXED>(L, R, guess, LEARNED || a.guess != nullptr, a, g, F, mine, !MUSCL,
                               sums);
    if (a.update && active && j > j0) {
      const int64_t off = base + (j - 1) * stride;
#pragma unroll
      for (int k = 0; k < NC; ++k)
        __builtin_nontemporal_store(Um[k] + dt_dx * (Fprev[k] - F[k]), &a.out[k][off]);
    }
    if constexpr (MUSCL) {
      if (a.check) CheckFace<D, DIR>(Um, U0, mine, a, g, crit, sums);
    }
    L = Lnext;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      Um[k] = U0[k];
      U0[k] = Up[k];
      Fprev[k] = F[k];
    }
  }
  BlockReduceGodunov<kBlock / 64>(sums.smax, a.dx, sums.iters, sums.max_it, sums.fails, sums.packed_faces(),
                                  a.partials + 5 * (blockIdx.x + static_cast<int64_t>(blockIdx.y) * gridDim.x));
}

// Reduction of the per-workgroup Godunov partials: out[0] = min dt,
// stats[0..3] = total iterations, max iterations, non-converged, faces.
// One workgroup per direction (partials of direction d at p + 5 n d, its
// minimum to out[d]); with `check` the value is also the split step's CFL
// check against ctl->split_dt.
constexpr int kRedBlock = 1024;
__global__ __launch_bounds__(kRedBlock) void GodunovFinalize(const unsigned long long* p,
                                                             int64_t n, double* out,
                                                             unsigned long long* stats, Ctl* ctl,
                                                             int check) {
  const int halt = ctl ? ctl->halt : 0;
  const double split_dt = check ? ctl->split_dt : 0.0;
  if (halt) return;
  p += 5 * n * blockIdx.x;
  __shared__ unsigned long long s[5][kRedBlock / 64];
  unsigned long long key = kInfKey, iters = 0, max_it = 0, fails = 0, faces = 0;
  // two blocks' partials a thread and round, loaded unconditionally
  for (int64_t i = threadIdx.x; i < n; i += 2 * kRedBlock) {
    const int64_t i2 = i + kRedBlock < n ? i + kRedBlock : i;
    unsigned long long v[2][5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      v[0][k] = p[5 * i + k];
      v[1][k] = p[5 * i2 + k];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (u == 1 && i2 == i) break;
      key = KMin(key, v[u][0]);
      iters += v[u][1];
      max_it = v[u][2] > max_it ? v[u][2] : max_it;
      fails += v[u][3];
      faces += v[u][4];
    }
  }
  key = WaveMinKey(key);
  iters = WaveSum(iters);
  max_it = WaveMaxU(max_it);
  fails = WaveSum(fails);
  faces = WaveSum(faces);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    s[0][wave] = key;
    s[1][wave] = iters;
    s[2][wave] = max_it;
    s[3][wave] = fails;
    s[4][wave] = faces;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < kRedBlock / 64; ++w) {
    key = KMin(key, s[0][w]);
    iters += s[1][w];
    max_it = s[2][w] > max_it ? s[2][w] : max_it;
    fails += s[3][w];
    faces += s[4][w];
  }
  const double v = __longlong_as_double(static_cast<long long>(key));
  if (out) out[blockIdx.x] = v;
  if (stats) {
    // faces packs the faces (low 32 bits) and the fallbacks (high bits)
    atomicAdd(&stats[0], iters);
    atomicMax(&stats[1], max_it);
    atomicAdd(&stats[2], fails);
    atomicAdd(&stats[3], faces & 0xffffffffull);
    atomicAdd(&stats[4], faces >> 32);
  }
  if (check && v < split_dt) {
    // TimeStepTooLarge{level_dt} (DimensionalSplitLevelIntegrator.hpp:243-245)
    ctl->halt = 1;
    ctl->failure_dt = v;
  }
}

// Per-face Godunov flux on strided views (FluxMethod seq driver): first
// order, or MUSCL-Hancock with the sequential (scalar) CompleteFromCons.
template <int D, int DIR>
__global__ __launch_bounds__(kBlock) void GodunovViewFlux(DevView fl, DevView st, double dt,
                                                          double dx, Gas<double> g, int limiter,
                                                          int muscl, double tol, int max_it,
                                                          unsigned long long* nfail) {
  using I = Idx<D>;
  constexpr int NC = D + 2, NQ = D + 4;
  const int64_t q = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (q >= fl.count()) return;
  int64_t f[3];
  fl.index(q, f);
  CellState<D> L, R;
  auto loadc = [&](int64_t off, double* out, int n) {
    int64_t c[3] = {f[0], f[1], f[2]};
    c[DIR] += off;
    for (int k = 0; k < n; ++k) out[k] = *st.at(c, k);
  };
  if (muscl) {
    const double y_g = NearArith::inv(g.gm1inv);
    double u[4][NC];
    for (int s = 0; s < 4; ++s) loadc(s - 2, u[s], NC);
    const double lh = 0.5 * dt / dx;
    CellState<D> unused;
    ReconAny<D, DIR, kRightState>(limiter, u[0], u[1], u[2], lh, g, y_g, unused, L);
    ReconAny<D, DIR, kLeftState>(limiter, u[1], u[2], u[3], lh, g, y_g, R, unused);
  } else {
    loadc(-1, L.q, NQ);
    loadc(0, R.q, NQ);
    L.y = NearArith::inv(L.q[0]);
    R.y = NearArith::inv(R.q[0]);
  }
  NewtonParams np;
  np.tol = tol;
  np.max_it = max_it;
  double uL, uR;
  FaceVelocities(L.q[1 + DIR], L.q[0], L.y, L.q[I::kA], R.q[1 + DIR], R.q[0], R.y, R.q[I::kA], &uL,
                 &uR);
  const MiddleState ms =
      SolveMiddleState(L.q[0], uL, L.q[I::kP], L.q[I::kA], R.q[0], uR, R.q[I::kP], R.q[I::kA], g,
                       np, 0.5 * (L.q[I::kP] + R.q[I::kP]));
  if (!ms.converged) atomicAdd(nfail, 1ull);
  double F[NC], wL, wR;
  GodunovSpeed(L.q[0], uL, L.q[I::kP], L.q[I::kA], R.q[0], uR, R.q[I::kP], R.q[I::kA], ms,
               g.gamma, &wL, &wR);
  GodunovFlux<D, DIR, false>(F, L.q, L.y, R.q, R.y, ms, wL, wR, g);
  for (int k = 0; k < NC; ++k) *fl.at(f, k) = F[k];
}

// Godunov::ComputeStableDt through the sequential driver: faces c in
// [lo, hi - S] with S = 2 * width; the base sees cells c + w - 1, c + w.
template <int D, int DIR>
__global__ __launch_bounds__(kBlock) void GodunovViewStableDt(DevView st, DevView faces, int w,
                                                              double dx, Gas<double> g,
                                                              double tol, int max_it,
                                                              unsigned long long* partials) {
  constexpr int NQ = D + 4;
  const int64_t q = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  unsigned long long key = kInfKey;
  if (q < faces.count()) {
    int64_t c[3];
    faces.index(q, c);
    c[DIR] += w - 1;
    double L[NQ], R[NQ];
    for (int k = 0; k < NQ; ++k) L[k] = *st.at(c, k);
    c[DIR] += 1;
    for (int k = 0; k < NQ; ++k) R[k] = *st.at(c, k);
    key = SpeedKey(dx, CellFaceSpeed<D>(L, L[1 + DIR], R, R[1 + DIR], g, tol, max_it, nullptr));
  }
  __shared__ unsigned long long s[kBlock / 64];
  key = WaveMinKey(key);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = key;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long k = s[0];
    for (int i = 1; i < kBlock / 64; ++i) k = KMin(k, s[i]);
    partials[blockIdx.x] = k;
  }
}

// Step-start CFL of all directions for the exact solver: the largest signal
// speed a direction, from the faces that can hold it.
//
// With a speed floor (floor[d] > 0, a lower bound of direction d's largest
// speed) a face is solved only when its certified bounds (QuickSpeedBelow for
// every face, SpeedBelow for those it leaves) reach the floor; blocks whose
// solved faces reach it set hit[d], which proves that the skipped ones are
// slower than the maximum.  Without a floor every face is
// solved, by the same instructions, so dt does not depend on the floor.
//
// 3D: a workgroup's eight waves are eight x rows of 64 cells marching along
// z; lanes 1..62 own their cells and lane 0 and row 0 are halos.  2D: each
// wave marches along y by itself.  A cell's six floats reach the x neighbour
// by DPP, the y neighbour through LDS (3D), the marching neighbour in
// registers; faces to be solved reload their cells.  Bound by the serial march
// (a step's loads and barriers) and 318 (smooth) to 380 (strong waves)
// instructions a cell, VALU busy 47%, next to one read of the state.  The kernel it
// replaces solved every face of the first sweep's direction, for that sweep's
// reuse, and every face outside a narrow class; solving them in the sweep
// alone costs less.  First-order step, 384^3 strong-wave blocks: 19.7 -> 11.0
// ms, mixed learned form at 203 x 149 x 121: 1.72 -> 1.06 ms.
constexpr int kCflRows = 8;
constexpr int kCflOwnX = 62;
constexpr int kCflBlocks = 4096;

struct GodunovCflArgs {
  const double* in[5];
  int64_t n[3];
  double dx[3];
  double gamma, gm1inv, tol;
  int max_it;
  SpeedBound bound;
  int64_t items;                 // tiles x segments
  int seg;                       // cells of a segment along the march
  unsigned long long* partials;  // 5 per workgroup and direction
  int* halt;
  const double* floor;  // speed floor per direction (nullable: none)
  int* hit;
  int count_fails;  // faces that hit the iteration cap count as failures (first
                    // order, where the sweeps solve the same faces)
};

// The face of direction d between the cells at off_l and off_r: its largest
// signal speed, from Newton.  Out of line: inlined, the solver's registers are
// the marching loop's spills (the pass at 384^3 on strong waves: 1103 us, out
// of line 1035).
struct CflFaceResult {
  double speed;
  int iterations, converged;
};
template <int D>
__device__ __attribute__((noinline)) CflFaceResult CflFace(const double* u0, const double* u1,
                                                           const double* u2, const double* u3,
                                                           const double* u4, double gamma,
                                                           double gm1inv, double tol, int max_it,
                                                           int d, int64_t off_l, int64_t off_r) {
  const double* in[5] = {u0, u1, u2, u3, u4};
  Gas<double> g;
  g.gamma = gamma;
  g.gm1inv = gm1inv;
  g.gm1 = gamma - 1.0;
  double L[D + 4], R[D + 4];
#pragma unroll
  for (int k = 0; k < D + 2; ++k) {
    L[k] = in[k][off_l];
    R[k] = in[k][off_r];
  }
  CompleteFromCons<D>(L, g);
  CompleteFromCons<D>(R, g);
  const double mL = d == 0 ? L[1] : (D == 2 || d == 1) ? L[2] : L[D];
  const double mR = d == 0 ? R[1] : (D == 2 || d == 1) ? R[2] : R[D];
  unsigned long long acc[3] = {0, 0, 0};
  CflFaceResult r;
  r.speed = CellFaceSpeed<D>(L, mL, R, mR, g, tol, max_it, acc);
  r.iterations = static_cast<int>(acc[0]);
  r.converged = acc[2] == 0;
  return r;
}

template <int D> __device__ __forceinline__ SpeedCell<D> ShiftUpCell(const SpeedCell<D>& c) {
  SpeedCell<D> r;
  r.ir = ShiftUp(c.ir);
  r.p = ShiftUp(c.p);
  r.a2 = ShiftUp(c.a2);
#pragma unroll
  for (int d = 0; d < D; ++d) r.u[d] = ShiftUp(c.u[d]);
  return r;
}

constexpr int kCflSeg = 32;  // cells of a segment along the march, at most

// SHORT: segments of a.seg cells (GodunovCflSeg), otherwise of kCflSeg.
template <int D, bool SHORT>
__global__ __launch_bounds__(64 * kCflRows) __attribute__((amdgpu_waves_per_eu(4))) void GodunovCflKernel(GodunovCflArgs a) {
  constexpr int NC = D + 2;
  const int seg_cells = SHORT ? a.seg : kCflSeg;
  constexpr int M = D - 1;  // marching direction
  if (a.halt && *a.halt) return;
  Gas<double> g;
  g.gamma = a.gamma;
  g.gm1inv = a.gm1inv;
  g.gm1 = a.gamma - 1.0;
  const int64_t nx = a.n[0], ny = a.n[1];
  const int64_t nm = a.n[M];
  const int64_t ms = (D == 3) ? nx * ny : nx;
  const int lane = threadIdx.x & 63;
  const int row = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  float F[3] = {0.0f, 0.0f, 0.0f};
  if (a.floor) {
#pragma unroll
    for (int d = 0; d < D; ++d) F[d] = static_cast<float>(a.floor[d] * (1.0 - 0x1p-20));
  }
  __shared__ SpeedCell<D> s_c[D == 3 ? 2 * kCflRows * 64 : 1];
  const int64_t tiles_x = (nx + kCflOwnX - 1) / kCflOwnX;
  const int64_t tiles_y = (D == 3) ? (ny + kCflRows - 2) / (kCflRows - 1) : 1;
  double smax[3] = {0.0, 0.0, 0.0};
  unsigned long long acc[3] = {0, 0, 0};  // iterations, largest, not converged
  unsigned faces[3] = {0, 0, 0};
  // Faces to solve wait in a list of the wave's until 64 of them fill it: the
  // few of a step (0.3% of the faces of strong-wave blocks) would each cost the
  // whole wave a Newton solve.  An entry is a cell and the face of it: d its
  // lower face of direction d, 4 + d a face that joins it with its own copy.
  // A step adds at most six entries a lane.
  __shared__ int64_t s_list[kCflRows][64 + 6 * 64];
  int64_t* list = s_list[row];
  int count = 0;  // wave-uniform
  auto solve = [&]() {
    const int n = count < 64 ? count : 64;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < n) {
      const int64_t entry = list[count - n + lane];
      const int d = static_cast<int>(entry & 3);
      const int64_t off = entry >> 3;
      const int64_t back = d == 0 ? 1 : d == M ? ms : nx;
      const CflFaceResult r =
          CflFace<D>(a.in[0], a.in[1], a.in[2], a.in[3], a.in[4], a.gamma, a.gm1inv, a.tol,
                     a.max_it, d, (entry & 4) ? off : off - back, off);
      const double v = r.speed;
      const unsigned long long it = static_cast<unsigned long long>(r.iterations);
      acc[0] += it;
      acc[1] = it > acc[1] ? it : acc[1];
      acc[2] += r.converged ? 0 : 1;
      faces[0] += d == 0;
      faces[1] += d == 1;
      faces[2] += d == 2;
      if (d == 0) smax[0] = __builtin_fmax(smax[0], v);
      if (d == 1) smax[1] = __builtin_fmax(smax[1], v);
      if (d == 2) smax[2] = __builtin_fmax(smax[2], v);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    count -= n;
  };
  // 3D: a block per item; 2D: a wave per item (uniform loops either way)
  const int64_t first = D == 3 ? blockIdx.x : static_cast<int64_t>(blockIdx.x) * kCflRows + row;
  const int64_t step = D == 3 ? gridDim.x : static_cast<int64_t>(gridDim.x) * kCflRows;
  int buf = 0;
  for (int64_t item = first; item < a.items; item += step) {
    const int64_t tx = item % tiles_x, ty = (item / tiles_x) % tiles_y;
    const int64_t seg = item / (tiles_x * tiles_y);
    const int64_t x = tx * kCflOwnX + lane - 1;
    const int64_t y = (D == 3) ? ty * (kCflRows - 1) + row - 1 : 0;
    const bool own = lane >= 1 && lane <= kCflOwnX && x < nx && (D == 2 || (row >= 1 && y < ny));
    const int64_t xs = Clamp(x, nx), ys = (D == 3) ? Clamp(y, ny) : 0;
    const int64_t col = xs + (D == 3 ? ys * nx : 0);
    const int64_t m0 = seg * seg_cells;
    const int64_t m1 = (m0 + seg_cells < nm) ? m0 + seg_cells : nm;
    auto load = [&](double* u, int64_t m) {
      const int64_t off = col + Clamp(m, nm) * ms;
#pragma unroll
      for (int k = 0; k < NC; ++k) u[k] = a.in[k][off];
    };
    double ucur[NC], unext[NC];
    load(ucur, m0 - 1);
    SpeedCell<D> cprev = MakeSpeedCell<D>(ucur, g);
    load(ucur, m0);
    for (int64_t m = m0; m < m1; ++m) {
      if (m + 1 < m1) load(unext, m + 1);
      const SpeedCell<D> c = MakeSpeedCell<D>(ucur, g);
      const SpeedCell<D> cl = ShiftUpCell<D>(c);
      // Faces to solve: bit d the cell's lower face of direction d, bit 4 + d
      // the patch's upper face, which joins a cell with its own copy.
      unsigned todo = 0;
      if constexpr (D == 3) {
        s_c[(buf * kCflRows + row) * 64 + lane] = c;
        __syncthreads();
      }
      // Every face takes the quick test; a wave with a face that does not pass
      // it (strong waves) takes the tight one.
      auto below = [&](const SpeedCell<D>& l, float ul, float ur, float f) {
        bool pass = !own || QuickSpeedBelow<D>(l, ul, c, ur, a.bound, f);
        if (__any(!pass)) pass = !own || SpeedBelow<D>(l, ul, c, ur, a.bound, f);
        return pass;
      };
      if (!below(cl, cl.u[0], c.u[0], F[0])) todo |= 1u;
      if constexpr (D == 3) {
        const SpeedCell<D> cb = s_c[(buf * kCflRows + (row > 0 ? row - 1 : 0)) * 64 + lane];
        if (!below(cb, cb.u[1], c.u[1], F[1])) todo |= 2u;
        if (own && y == ny - 1 && !QuickSpeedBelow<D>(c, c.u[1], c, c.u[1], a.bound, F[1]))
          todo |= 32u;
      }
      if (!below(cprev, cprev.u[M], c.u[M], F[M])) todo |= 1u << M;
      if (own) {
        if (x == nx - 1 && !QuickSpeedBelow<D>(c, c.u[0], c, c.u[0], a.bound, F[0])) todo |= 16u;
        if (m == nm - 1 && !QuickSpeedBelow<D>(c, c.u[M], c, c.u[M], a.bound, F[M]))
          todo |= 16u << M;
      }
      buf ^= 1;
      if (__builtin_expect(__any(todo != 0), 0)) {
        const int64_t off = col + m * ms;
        // the patch's lower faces join a cell with its own copy, too
        const unsigned edge = (x <= 0 ? 1u : 0u) | (D == 3 && y <= 0 ? 2u : 0u) |
                              (m == 0 ? 1u << M : 0u);
        todo = (todo & ~edge) | ((todo & edge) << 4);
        for (int f = 0; f < 7; ++f) {
          const bool mine = (todo >> f) & 1u;
          const unsigned long long who = __ballot(mine);
          if (mine)
            list[count + __builtin_popcountll(who & ((1ull << lane) - 1ull))] = (off << 3) | f;
          count += static_cast<int>(__builtin_popcountll(who));
        }
        while (count >= 64) solve();
      }
      cprev = c;
#pragma unroll
      for (int k = 0; k < NC; ++k) ucur[k] = unext[k];
    }
  }
  while (count > 0) solve();
  // The iteration counters of all directions go with direction 0's partials.
  const int64_t nblocks = gridDim.x;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const bool first_dir = d == 0;
    BlockReduceGodunov<kCflRows>(smax[d], a.dx[d], first_dir ? acc[0] : 0, first_dir ? acc[1] : 0,
                                 first_dir && a.count_fails ? acc[2] : 0, faces[d],
                                 a.partials + 5 * (d * nblocks + blockIdx.x));
    const bool hit = a.floor && a.floor[d] > 0.0 && smax[d] >= a.floor[d];
    if (__syncthreads_or(hit ? 1 : 0) && threadIdx.x == 0 && a.hit) a.hit[d] = 1;
  }
}

// Speed floor of a state the level knows nothing about yet (its first step):
// the largest |u| + a of the cells, a lower bound of the largest signal speed
// of direction d because each cell is the right state of one face and the left
// state of the next (uR + aR or more where u >= 0, |uL| + aL or more where u <
// 0).  Reads the state once; without it the first pass solves every face
// (three Newton solves a cell).  cfl_floor[d] grows by an atomic maximum (non-
// negative doubles order like their bits), on top of a caller's hint.
template <int D>
__global__ __launch_bounds__(kBlock) void GodunovFloorKernel(GodunovCflArgs a, int64_t ncell,
                                                             Ctl* ctl) {
  if (ctl->halt || ctl->floor_known) return;
  Gas<double> g;
  g.gamma = a.gamma;
  g.gm1inv = a.gm1inv;
  g.gm1 = a.gamma - 1.0;
  double s[D];
#pragma unroll
  for (int d = 0; d < D; ++d) s[d] = 0.0;
  const int64_t step = static_cast<int64_t>(gridDim.x) * kBlock;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < ncell; i += step) {
    double q[D + 4];
#pragma unroll
    for (int k = 0; k < D + 2; ++k) q[k] = a.in[k][i];
    const double y = NearArith::inv(q[0]);
    const double p = (q[D + 1] - 0.5 * SqNormArray<D>(q + 1) * y) * g.gm1;
    if (q[0] > 0.0 && p > 0.0) {
      const double c = NearArith::sqrt(g.gamma * p * y);
#pragma unroll
      for (int d = 0; d < D; ++d) s[d] = __builtin_fmax(s[d], rabs(q[1 + d] * y) + c);
    }
  }
  __shared__ double sh[D][kBlock / 64];
#pragma unroll
  for (int d = 0; d < D; ++d) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s[d] = __builtin_fmax(s[d], __shfl_xor(s[d], off, 64));
    if ((threadIdx.x & 63) == 0) sh[d][threadIdx.x >> 6] = s[d];
  }
  __syncthreads();
  if (threadIdx.x < D) {
    double v = sh[threadIdx.x][0];
    for (int w = 1; w < kBlock / 64; ++w) v = __builtin_fmax(v, sh[threadIdx.x][w]);
    v *= 1.0 - 0x1p-20;
    if (v > 0.0 && v < 1.7976931348623157e308)
      atomicMax(reinterpret_cast<unsigned long long*>(&ctl->cfl_floor[threadIdx.x]),
                static_cast<unsigned long long>(__double_as_longlong(v)));
  }
}

// ComputeMiddleState on arrays of complete state pairs (SoA (D+4) x n) with
// optional initial guesses; pM, uM, iterations and convergence per pair.
template <int D>
__global__ __launch_bounds__(kBlock) void MiddleStateKernel(const double* __restrict__ L,
                                                            const double* __restrict__ R,
                                                            int64_t n, int dir, double gamma,
                                                            double tol, int max_it,
                                                            const double* __restrict__ guess,
                                                            double* pM, double* uM, int* iters,
                                                            int* conv) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  double l[D + 4], r[D + 4];
  for (int k = 0; k < D + 4; ++k) {
    l[k] = L[k * n + i];
    r[k] = R[k * n + i];
  }
  Gas<double> g;
  g.gamma = gamma;
  g.gm1inv = 1.0 / (gamma - 1.0);
  g.gm1 = gamma - 1.0;
  NewtonParams np;
  np.tol = tol;
  np.max_it = max_it;
  const double x0 = guess ? guess[i] : 0.5 * (l[D + 2] + r[D + 2]);
  MiddleState ms;
  if (dir == 0) ms = ComputeMiddleState<D, 0>(l, r, g, np, x0);
  else if (dir == 1) ms = ComputeMiddleState<D, 1>(l, r, g, np, x0);
  else ms = ComputeMiddleState<D, (D > 2 ? 2 : 0)>(l, r, g, np, x0);
  if (pM) pM[i] = ms.pM;
  if (uM) uM[i] = ms.uM;
  if (iters) iters[i] = ms.iterations;
  if (conv) conv[i] = ms.converged;
}

} // namespace

int LaunchMiddleState(int dim, hipStream_t s, const double* L, const double* R, int64_t n,
                      int dir, double gamma, double tol, int max_it, const double* guess,
                      double* pM, double* uM, int* iters, int* conv) {
  const unsigned blocks = unsigned((n + kBlock - 1) / kBlock);
  if (dim == 2)
    hipLaunchKernelGGL(MiddleStateKernel<2>, dim3(blocks), dim3(kBlock), 0, s, L, R, n, dir, gamma,
                       tol, max_it, guess, pM, uM, iters, conv);
  else
    hipLaunchKernelGGL(MiddleStateKernel<3>, dim3(blocks), dim3(kBlock), 0, s, L, R, n, dir, gamma,
                       tol, max_it, guess, pM, uM, iters, conv);
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

// Segment of a pencil sweep: PencilSeg, longer where the grid's second
// dimension (65,535) would not hold its segments.
static int GodunovSeg(int dim, int dir, const int64_t n[3]) {
  int64_t seg = PencilSeg(dim, dir, n);
  while ((n[dir] + seg - 1) / seg > 65535) seg *= 2;
  return static_cast<int>(seg);
}

int64_t GodunovSweepBlocks(int dim, int dir, const int64_t n[3]) {
  return SweepBlocks(dim, dir, n, GodunovSeg(dim, dir, n));
}

// Cells of a segment of the CFL pass: 32, halved down to 1 while the items are
// too few to fill the chip (3D: 256 workgroups of eight waves, 2D: 1,024
// waves).  A segment is a serial chain of loads and barriers, and a row more is
// loaded per segment.  First-order step, us, with 32 cells always and with this
// rule: 16^2 76, 57; 256^2 114, 62; 1000^2 227, 174; 32^3 194, 79; 64^3 285,
// 142; 96^3 362, 239; 128^3 490, 419 (512 waves in 2D: 1000^2 227; 512
// workgroups in 3D: 64^3 151, 128^3 404, and 203 x 149 x 121 in strong waves,
// 352 workgroups of whole segments, 4.23 -> 4.32 ms for four steps).
static int GodunovCflSeg(int64_t nm, int64_t tiles, int64_t enough) {
  int seg = kCflSeg;
  while (seg > 1 && tiles * ((nm + seg - 1) / seg) < enough) seg /= 2;
  return seg;
}

static int64_t GodunovCflItems(int dim, const int64_t n[3], int* seg = nullptr) {
  const int64_t tx = (n[0] + kCflOwnX - 1) / kCflOwnX;
  const int64_t ty = dim == 3 ? (n[1] + kCflRows - 2) / (kCflRows - 1) : 1;
  const int64_t nm = dim == 3 ? n[2] : n[1];
  const int s = GodunovCflSeg(nm, tx * ty, dim == 3 ? 256 : 1024);
  if (seg) *seg = s;
  return tx * ty * ((nm + s - 1) / s);
}

int64_t GodunovCflBlocks(int dim, const int64_t n[3]) {
  const int64_t items = GodunovCflItems(dim, n);
  const int64_t blocks = dim == 3 ? items : (items + kCflRows - 1) / kCflRows;
  return blocks < kCflBlocks ? blocks : kCflBlocks;
}

int LaunchGodunovSweep(const fvs_method_desc& desc, hipStream_t s, int dir,
                       const double* const* in, double* const* out, const int64_t n[3],
                       double dx, const double* dt_ptr, double dt_val, const double* guess,
                       unsigned long long* partials, int* halt, int update,
                       const fvs_mlp* net, int check) {
  GodunovArgs a;
  std::memset(&a, 0, sizeof a);
  const int D = desc.dim;
  for (int c = 0; c < D + 2; ++c) {
    a.in[c] = in[c];
    a.out[c] = out ? out[c] : nullptr;
  }
  for (int d = 0; d < 3; ++d) a.n[d] = (d < D) ? n[d] : 1;
  a.dx = dx;
  a.dt_ptr = dt_ptr;
  a.dt_val = dt_val;
  a.gamma = desc.gamma;
  a.gm1inv = 1.0 / (desc.gamma - 1.0);
  a.tol = desc.newton_tolerance;
  a.max_it = desc.max_newton_iterations;
  a.guess = guess;
  if (net) MlpOperands(net, &a.tiles, &a.bias);
  a.partials = partials;
  a.halt = halt;
  a.seg = GodunovSeg(D, dir, a.n);
  a.update = update;
  const bool muscl = desc.reconstruction == FVS_RECON_MUSCL_HANCOCK;
  a.limiter = desc.limiter;
  a.check = check;
  a.bound = MakeSpeedBound(desc.gamma, desc.newton_tolerance, desc.max_newton_iterations);
  const bool mixed = desc.precision == FVS_FP32_FLUX;
  const bool learned = a.tiles != nullptr;
  if (muscl && (learned || guess)) {
    SetError("MUSCL-Hancock sweeps take no guess");
    return FVS_BAD_ARGUMENT;
  }
  const int64_t blocks = GodunovSweepBlocks(D, dir, a.n);
  if (blocks <= 0) return FVS_BAD_ARGUMENT;
  if (dir == 0) {
    if ((a.n[0] + 2) * a.n[1] * a.n[2] >= (int64_t(1) << 32)) {
      SetError("Godunov X sweep: patch too large for 32-bit slot indices");
      return FVS_BAD_ARGUMENT;
    }
    using K = void (*)(GodunovArgs);
#define FVS_GX(D_, LONG_)                                                                          \
  {                                                                                                \
    {GodunovSweepX<D_, false, false, false, LONG_>, GodunovSweepX<D_, false, true, false, LONG_>}, \
    {GodunovSweepX<D_, true, false, false, LONG_>, GodunovSweepX<D_, true, true, false, LONG_>}    \
  }
    const K ks[2][2][2][2] = {{FVS_GX(2, false), FVS_GX(3, false)}, {FVS_GX(2, true), FVS_GX(3, true)}};
#undef FVS_GX
    const K km[2][2] = {
        {GodunovSweepX<2, false, false, true, false>, GodunovSweepX<3, false, false, true, false>},
        {GodunovSweepX<2, false, false, true, true>, GodunovSweepX<3, false, false, true, true>}};
    const int lr = a.n[0] >= kXLongRow;
    hipLaunchKernelGGL(muscl ? km[lr][D == 3] : ks[lr][D == 3][mixed][learned],
                       dim3(unsigned(blocks)), dim3(kBlock), 0, s, a);
  } else {
    const int64_t npencil = (dir == 1) ? a.n[0] * a.n[2] : a.n[0] * a.n[1];
    const int64_t bx = (npencil + kBlock - 1) / kBlock;
    const int64_t nseg = (a.n[dir] + a.seg - 1) / a.seg;
    if (bx > 0x7fffffff || nseg > 65535) return FVS_BAD_ARGUMENT;
    const dim3 grid{static_cast<unsigned>(bx), static_cast<unsigned>(nseg), 1u};
    using K = void (*)(GodunovArgs);
#define FVS_GP(D_, R_)                                                                          \
  {                                                                                             \
    {GodunovSweepPencil<D_, R_, false, false, false>, GodunovSweepPencil<D_, R_, false, true, false>}, \
    {GodunovSweepPencil<D_, R_, true, false, false>, GodunovSweepPencil<D_, R_, true, true, false>} \
  }
    const K ks[3][2][2] = {FVS_GP(2, 1), FVS_GP(3, 1), FVS_GP(3, 2)};
#undef FVS_GP
    const K km[3] = {GodunovSweepPencil<2, 1, false, false, true>,
                     GodunovSweepPencil<3, 1, false, false, true>,
                     GodunovSweepPencil<3, 2, false, false, true>};
    const int which = D == 2 ? 0 : (dir == 1 ? 1 : 2);
    hipLaunchKernelGGL(muscl ? km[which] : ks[which][mixed][learned], grid, dim3(kBlock), 0, s, a);
  }
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

int LaunchGodunovFinalize(hipStream_t s, const unsigned long long* partials, int64_t nblocks,
                          int ndir, double* out, unsigned long long* stats, Ctl* ctl, int check) {
  hipLaunchKernelGGL(GodunovFinalize, dim3(ndir), dim3(kRedBlock), 0, s, partials, nblocks, out,
                     stats, ctl, check);
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

int LaunchGodunovCfl(const fvs_method_desc& desc, hipStream_t s, const double* const* cons,
                     const int64_t n[3], const double dx[3], unsigned long long* partials,
                     int* halt, Ctl* floor_ctl) {
  GodunovCflArgs a;
  std::memset(&a, 0, sizeof a);
  const int D = desc.dim;
  for (int c = 0; c < D + 2; ++c) a.in[c] = cons[c];
  int64_t ncell = 1;
  for (int d = 0; d < 3; ++d) {
    a.n[d] = (d < D) ? n[d] : 1;
    a.dx[d] = (d < D) ? dx[d] : 1.0;
    ncell *= a.n[d];
  }
  a.gamma = desc.gamma;
  a.gm1inv = 1.0 / (desc.gamma - 1.0);
  a.tol = desc.newton_tolerance;
  a.max_it = desc.max_newton_iterations;
  a.bound = MakeSpeedBound(desc.gamma, desc.newton_tolerance, desc.max_newton_iterations);
  a.items = GodunovCflItems(D, a.n, &a.seg);
  a.count_fails = desc.reconstruction == FVS_RECON_NONE;
  a.partials = partials;
  a.halt = halt;
  const dim3 grid(static_cast<unsigned>(GodunovCflBlocks(D, a.n)));
  const dim3 block(64 * kCflRows);
  if (floor_ctl && desc.max_newton_iterations >= kGodunovFloorCap) {
    a.floor = floor_ctl->cfl_floor;
    a.hit = floor_ctl->floor_hit;
    const int64_t fb = (ncell + kBlock - 1) / kBlock;
    const dim3 fgrid(static_cast<unsigned>(fb < 2048 ? fb : 2048));
    if (D == 3)
      hipLaunchKernelGGL(GodunovFloorKernel<3>, fgrid, dim3(kBlock), 0, s, a, ncell, floor_ctl);
    else
      hipLaunchKernelGGL(GodunovFloorKernel<2>, fgrid, dim3(kBlock), 0, s, a, ncell, floor_ctl);
    FVS_LAUNCH_CHECK();
  }
  using K = void (*)(GodunovCflArgs);
  const K ks[2][2] = {{GodunovCflKernel<2, false>, GodunovCflKernel<2, true>},
                      {GodunovCflKernel<3, false>, GodunovCflKernel<3, true>}};
  hipLaunchKernelGGL(ks[D == 3][a.seg < kCflSeg], grid, block, 0, s, a);
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

static int MakeGView(const fvs_view* v, DevView* out) { return MakeDevView(v, 1, out); }

int LaunchGodunovViewFlux(const fvs_method_desc& desc, hipStream_t s, const fvs_view* fluxes,
                          const fvs_view* states, double dt, double dx, int dir,
                          unsigned long long* nfail) {
  DevView fl, st;
  if (MakeGView(fluxes, &fl) || MakeGView(states, &st)) return FVS_BAD_ARGUMENT;
  Gas<double> g;
  g.gamma = desc.gamma;
  g.gm1inv = 1.0 / (desc.gamma - 1.0);
  g.gm1 = desc.gamma - 1.0;
  const int muscl = desc.reconstruction == FVS_RECON_MUSCL_HANCOCK;
  const unsigned nb = unsigned((fl.count() + kBlock - 1) / kBlock);
#define FVS_GVF(DD, DR)                                                                      \
  hipLaunchKernelGGL((GodunovViewFlux<DD, DR>), dim3(nb), dim3(kBlock), 0, s, fl, st, dt, dx, g, \
                     desc.limiter, muscl, desc.newton_tolerance, desc.max_newton_iterations,  \
                     nfail)
  if (desc.dim == 2) {
    if (dir == 0) FVS_GVF(2, 0); else FVS_GVF(2, 1);
  } else {
    if (dir == 0) FVS_GVF(3, 0); else if (dir == 1) FVS_GVF(3, 1); else FVS_GVF(3, 2);
  }
#undef FVS_GVF
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

int64_t GodunovViewStableDtBlocks(const fvs_method_desc& desc, const fvs_view* states, int dir) {
  const int S = desc.reconstruction == FVS_RECON_MUSCL_HANCOCK ? 4 : 2;
  int64_t cnt = 1;
  for (int d = 0; d < 3; ++d) {
    int64_t e = states->hi[d] - states->lo[d] + 1;
    if (d == dir) e -= S;
    if (e <= 0) return 0;
    cnt *= e;
  }
  return (cnt + kBlock - 1) / kBlock;
}

int LaunchGodunovViewStableDt(const fvs_method_desc& desc, hipStream_t s, const fvs_view* states,
                              double dx, int dir, unsigned long long* partials) {
  DevView st;
  if (MakeGView(states, &st)) return FVS_BAD_ARGUMENT;
  const int w = desc.reconstruction == FVS_RECON_MUSCL_HANCOCK ? 2 : 1;
  DevView faces = st;
  faces.ext[dir] -= 2 * w;  // sequential driver: Shrink(box, dir, {0, StencilSize})
  if (faces.ext[dir] <= 0) return FVS_BAD_ARGUMENT;
  Gas<double> g;
  g.gamma = desc.gamma;
  g.gm1inv = 1.0 / (desc.gamma - 1.0);
  g.gm1 = desc.gamma - 1.0;
  const unsigned nb = unsigned((faces.count() + kBlock - 1) / kBlock);
#define FVS_GVD(DD, DR)                                                                       \
  hipLaunchKernelGGL((GodunovViewStableDt<DD, DR>), dim3(nb), dim3(kBlock), 0, s, st, faces, w, \
                     dx, g, desc.newton_tolerance, desc.max_newton_iterations, partials)
  if (desc.dim == 2) {
    if (dir == 0) FVS_GVD(2, 0); else FVS_GVD(2, 1);
  } else {
    if (dir == 0) FVS_GVD(3, 0); else if (dir == 1) FVS_GVD(3, 1); else FVS_GVD(3, 2);
  }
#undef FVS_GVD
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

} // namespace fvs
