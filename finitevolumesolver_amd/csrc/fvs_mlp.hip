// Learned initial guess for the exact Riemann solver's Newton iteration.
//
// A 6 -> 64 -> 64 -> 1 ReLU MLP maps a state pair to the log of the star
// pressure relative to sqrt(pL pR):
//   features  x = (ln rhoL s, uL / 5, ln pL s, ln rhoR s, uR / 5, ln pR s),
//             s = 1 / ln(1000)
//   output    r,  initial guess p0 = exp(0.5 (ln pL + ln pR) + r)
// Inference runs on the matrix cores: BF16 operands, FP32 accumulation,
// v_mfma_f32_16x16x16_bf16.  Activations are kept transposed (hidden units x
// faces) so that a layer's 16x16 accumulator tile has exactly the lane and
// element layout of the next layer's B operand (no data movement between
// layers).  Training (forward, backward, Adam) is FP32 throughout, its
// products on the matrix cores' FP32 instruction; labels come from the FP64 Newton iteration itself.  The Newton iteration that
// refines the guess is unchanged (include/fub/NewtonIteration.hpp:28-52).
#include "fvs_internal.hpp"
#include "fvs_mlp_infer.hpp"
#include "fvs_riemann.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

namespace fvs {

namespace {

using namespace mlp;

constexpr int kBlock = 256;

// Packs the FP32 master parameters into bf16 A-operand tiles and a bias
// vector (b1, b2, b3).
__global__ void MlpPackKernel(const float* __restrict__ p, short* __restrict__ tiles,
                              float* __restrict__ bias) {
  const int t = blockIdx.x;      // tile
  const int lane = threadIdx.x;  // 0..63
  const int i = lane & 15;
  for (int e = 0; e < 4; ++e) {
    const int k = (lane >> 4) * 4 + e;
    float v = 0.0f;
    if (t < 4) {
      const int out = t * 16 + i;
      v = (k < kIn) ? p[kOffW1 + out * kInPad + k] : 0.0f;
    } else if (t < 20) {
      const int m = (t - 4) / 4, kb = (t - 4) % 4;
      v = p[kOffW2 + (m * 16 + i) * kH + kb * 16 + k];
    } else {
      const int kb = t - 20;
      v = (i == 0) ? p[kOffW3 + kb * 16 + k] : 0.0f;
    }
    tiles[(t * 64 + lane) * 4 + e] = ToBf16(v);
  }
  if (t == 0) {
    for (int j = lane; j < 2 * kH + 1; j += 64) {
      bias[j] = (j < kH) ? p[kOffB1 + j] : (j < 2 * kH ? p[kOffB2 + j - kH] : p[kOffB3]);
    }
  }
}

// Inference on arrays of complete state pairs (SoA (D+4) x n).  Writes the
// network output r and the initial guess.
template <int D>
__global__ __launch_bounds__(kBlock) void MlpInferPairs(const double* __restrict__ L,
                                                        const double* __restrict__ R, int64_t n,
                                                        int dir, const short* __restrict__ tiles,
                                                        const float* __restrict__ bias,
                                                        float* __restrict__ r_out,
                                                        double* __restrict__ guess) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  const int64_t j = i < n ? i : n - 1;
  double l[D + 4], r[D + 4];
  for (int k = 0; k < D + 4; ++k) {
    l[k] = L[k * n + j];
    r[k] = R[k * n + j];
  }
  float x[kIn];
  Features<D>(l, r, dir, x);
  const float out = MlpWave(x, tiles, bias);
  if (i < n) {
    if (r_out) r_out[i] = out;
    if (guess) {
      const bool weak = WeakPair(l[0], l[1 + dir] / l[0], l[D + 2], l[D + 3], r[0],
                                 r[1 + dir] / r[0], r[D + 2], r[D + 3]);
      guess[i] = weak ? 0.5 * (l[D + 2] + r[D + 2]) : GuessFromOutput(l[D + 2], r[D + 2], out);
    }
  }
}

// Guesses for every face of direction DIR of a ghost-free transmissive patch
// (face box n with n[DIR] + 1, x fastest): the first-order Godunov states of
// face f are the (clamped) cells f - 1 and f.
template <int D, int DIR>
__global__ __launch_bounds__(kBlock) void MlpInferFaces(
    const double* __restrict__ u0, const double* __restrict__ u1, const double* __restrict__ u2,
    const double* __restrict__ u3, const double* __restrict__ u4, int64_t nx, int64_t ny,
    int64_t nz, double gamma, double gm1inv, const short* __restrict__ tiles,
    const float* __restrict__ bias, double* __restrict__ guess) {
  const double* in[5] = {u0, u1, u2, u3, u4};
  const int64_t fx = nx + (DIR == 0), fy = ny + (DIR == 1), fz = nz + (DIR == 2);
  const int64_t nf = fx * fy * fz;
  const int64_t q = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  const int64_t qq = q < nf ? q : nf - 1;
  int64_t c[3] = {qq % fx, (qq / fx) % fy, qq / (fx * fy)};
  const int64_t n3[3] = {nx, ny, nz};
  Gas<double> g;
  g.gamma = gamma;
  g.gm1inv = gm1inv;
  g.gm1 = gamma - 1.0;
  double L[D + 4], R[D + 4];
  int64_t cl[3] = {c[0], c[1], c[2]}, cr[3] = {c[0], c[1], c[2]};
  cl[DIR] = c[DIR] - 1 < 0 ? 0 : c[DIR] - 1;
  cr[DIR] = c[DIR] >= n3[DIR] ? n3[DIR] - 1 : c[DIR];
  const int64_t ol = cl[0] + nx * (cl[1] + ny * cl[2]);
  const int64_t orr = cr[0] + nx * (cr[1] + ny * cr[2]);
  for (int k = 0; k < D + 2; ++k) {
    L[k] = in[k][ol];
    R[k] = in[k][orr];
  }
  CompleteFromCons<D>(L, g);
  CompleteFromCons<D>(R, g);
  const bool weak = WeakPair(L[0], L[1 + DIR] / L[0], L[D + 2], L[D + 3], R[0],
                             R[1 + DIR] / R[0], R[D + 2], R[D + 3]);
  double p0 = 0.5 * (L[D + 2] + R[D + 2]);
  if (__ballot(!weak) != 0) {  // wave-uniform: skip the network when every face is weak
    float x[kIn];
    Features<D>(L, R, DIR, x);
    const float out = MlpWave(x, tiles, bias);
    if (!weak) p0 = GuessFromOutput(L[D + 2], R[D + 2], out);
  }
  if (q < nf) guess[q] = p0;
}

// ---- training ---------------------------------------------------------------

__device__ __forceinline__ uint64_t SplitMix(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
__device__ __forceinline__ double Uniform(uint64_t seed, uint64_t i, int k) {
  return static_cast<double>(SplitMix(seed ^ SplitMix(i * 8 + k)) >> 11) * (1.0 / 9007199254740992.0);
}

// Sample i: rho, p log-uniform in [1e-3, 1e3], u uniform in [-5, 5] on both
// sides; vacuum-generating pairs (2 aL / (g-1) + 2 aR / (g-1) <= uR - uL)
// are flagged; the label is the FP64 Newton star pressure (default guess).
// prim: 6 x n doubles (rhoL, uL, pL, rhoR, uR, pR); x: 6 x n floats;
// target: r = ln p* - 0.5 (ln pL + ln pR); flag: 0 ok, 1 vacuum, 2 no convergence.
__global__ __launch_bounds__(kBlock) void MlpSampleKernel(int64_t n, uint64_t seed, double gamma,
                                                          int max_it, double tol,
                                                          double* __restrict__ prim,
                                                          float* __restrict__ x,
                                                          float* __restrict__ target,
                                                          int* __restrict__ flag,
                                                          int* __restrict__ iters) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const double lo = log(1e-3), hi = log(1e3);
  const double rhoL = exp(lo + (hi - lo) * Uniform(seed, i, 0));
  const double uL = -5.0 + 10.0 * Uniform(seed, i, 1);
  const double pL = exp(lo + (hi - lo) * Uniform(seed, i, 2));
  const double rhoR = exp(lo + (hi - lo) * Uniform(seed, i, 3));
  const double uR = -5.0 + 10.0 * Uniform(seed, i, 4);
  const double pR = exp(lo + (hi - lo) * Uniform(seed, i, 5));
  const double pr[6] = {rhoL, uL, pL, rhoR, uR, pR};
  for (int k = 0; k < 6; ++k) prim[k * n + i] = pr[k];
  Gas<double> g;
  g.gamma = gamma;
  g.gm1inv = 1.0 / (gamma - 1.0);
  g.gm1 = gamma - 1.0;
  // Complete states (1D momentum along x; 2D layout with zero transverse).
  double L[6], R[6];
  auto complete = [&](double rho, double u, double p, double* q) {
    q[0] = rho;
    q[1] = rho * u;
    q[2] = 0.0;
    const double e_kin = 0.5 * (q[1] * q[1] + q[2] * q[2]) / rho;
    q[3] = e_kin + p * g.gm1inv;
    q[4] = p;
    q[5] = sqrt(gamma * p / rho);
  };
  complete(rhoL, uL, pL, L);
  complete(rhoR, uR, pR, R);
  float xf[kIn];
  Features<2>(L, R, 0, xf);
  for (int k = 0; k < kIn; ++k) x[k * n + i] = xf[k];
  const double gm1 = gamma - 1.0;
  if (2.0 * L[5] / gm1 + 2.0 * R[5] / gm1 <= uR - uL) {
    flag[i] = 1;
    target[i] = 0.0f;
    iters[i] = 0;
    return;
  }
  NewtonParams np;
  np.tol = tol;
  np.max_it = max_it;
  const MiddleState ms = ComputeMiddleState<2, 0>(L, R, g, np, 0.5 * (pL + pR));
  iters[i] = ms.iterations;
  if (!ms.converged || !(ms.pM > 0.0)) {
    flag[i] = 2;
    target[i] = 0.0f;
    return;
  }
  flag[i] = 0;
  target[i] = static_cast<float>(log(ms.pM) - 0.5 * (log(pL) + log(pR)));
}

// FP32 forward of one sample per thread.  x: 6 x n, y: n.
__global__ __launch_bounds__(kBlock) void MlpForwardKernel(const float* __restrict__ p,
                                                           const float* __restrict__ x, int64_t n,
                                                           float* __restrict__ y) {
  __shared__ float sp[kNParams];
  for (int k = threadIdx.x; k < kNParams; k += kBlock) sp[k] = p[k];
  __syncthreads();
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  float xi[kIn];
  for (int k = 0; k < kIn; ++k) xi[k] = x[k * n + i];
  float a1[kH];
  for (int o = 0; o < kH; ++o) {
    float s = sp[kOffB1 + o];
    for (int k = 0; k < kIn; ++k) s += sp[kOffW1 + o * kInPad + k] * xi[k];
    a1[o] = fmaxf(s, 0.0f);
  }
  float out = sp[kOffB3];
  for (int o = 0; o < kH; ++o) {
    float s = sp[kOffB2 + o];
    for (int k = 0; k < kH; ++k) s += sp[kOffW2 + o * kH + k] * a1[k];
    const float a2 = fmaxf(s, 0.0f);
    out += sp[kOffW3 + o] * a2;
  }
  y[i] = out;
}

// Loss and parameter gradients of a batch on the matrix cores, in FP32
// (v_mfma_f32_16x16x4_f32: FP32 operands, products and sums).
//
// A workgroup takes tiles of 16 samples, its four waves 16 hidden units each:
//   H1 = relu(W1 X + b1), H2 = relu(W2 H1 + b2), y = W3 H2 + b3,
//   loss e^2 (or the Huber form 2 h |e| - h^2 beyond |e| > h when huber h > 0)
//   over samples with flag 0, e = y - t, dy = 2 clamp(e, -h, h) inv_count,
//   dH2 = W3 dy [H2 > 0], dH1 = W2^T dH2 [H1 > 0],
//   gradients dW2 = dH2 H1^T, dW1 = dH1 X^T, biases and dW3 the row sums.
// The parameters sit in LDS and activations pass between the waves through
// it; the gradient tiles stay in accumulators over the workgroup's tiles and
// leave as one partial vector (part[block][kNParams]) that MlpReduceKernel
// sums in a fixed order, so training is deterministic.
//
// Operand layouts of the 16x16x4 product: A[i][k] and B[k][j] one value a
// lane (i or j = lane % 16, k = lane / 16), D[i][j] in lane j + 16 (i / 4),
// element i % 4.  The order of the summation index is free: step s of a
// 64-long sum takes index 16 k + s, so that LDS rows of 17 (and 65) floats are
// read without bank conflicts.
//
// A batch of 1,024 is 64 workgroups of 13 MFLOP together: latency bound.
// Three kernels of one sample (or one parameter) a thread, four and sixteen
// workgroups, took 41 + 87 + 145 us here; this one and the reduction take
// 11 + 3 us, and an epoch over 2^17 pairs 35.2 -> 2.6 ms with its data
// generation.
constexpr int kTile = 16;         // samples per tile
constexpr int kActStride = 17;    // LDS floats per activation row
constexpr int kW2Stride = 65;
static_assert(kBlock % kInPad == 0, "a thread stages one column of W1");
constexpr int kGradBlocks = 512;  // most workgroups (partial vectors)

__device__ __forceinline__ floatx4_t MfmaF32(float a, float b, floatx4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float RowSum16(float v) {  // over the 16 lanes of a row
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__global__ __launch_bounds__(kBlock) void MlpGradKernel(
    const float* __restrict__ p, const float* __restrict__ x, const float* __restrict__ t,
    const int* __restrict__ flag, int64_t n, const uint32_t* __restrict__ idx, int64_t nb,
    float inv_count, float huber, float* __restrict__ part, float* __restrict__ loss_part) {
  __shared__ float s_w1[kH * 9], s_w2[kH * kW2Stride], s_b1[kH], s_b2[kH], s_w3[kH];
  __shared__ float s_x[kInPad][kActStride];
  __shared__ float s_h1[kH][kActStride], s_d2[kH][kActStride], s_d1[kH][kActStride];
  __shared__ float s_y[4][kTile], s_dy[kTile], s_t[kTile];
  __shared__ int s_ok[kTile];
  // W1's padding columns, which a caller may have set to anything, meet the row
  // of ones below
  const bool input = threadIdx.x % kInPad < kIn;
  for (int k = threadIdx.x; k < kH * kInPad; k += kBlock) {
    const float v = p[kOffW1 + k];
    s_w1[(k / kInPad) * 9 + k % kInPad] = input ? v : 0.0f;
  }
  for (int k = threadIdx.x; k < kH * kH; k += kBlock)
    s_w2[(k / kH) * kW2Stride + k % kH] = p[kOffW2 + k];
  if (threadIdx.x < kH) {
    s_b1[threadIdx.x] = p[kOffB1 + threadIdx.x];
    s_b2[threadIdx.x] = p[kOffB2 + threadIdx.x];
    s_w3[threadIdx.x] = p[kOffW3 + threadIdx.x];
  }
  const float b3 = p[kOffB3];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;  // this wave's hidden units 16 w .. 16 w + 15
  const int q = lane >> 4, j = lane & 15;
  const int row = 16 * w + 4 * q;  // accumulator rows row .. row + 3, column j
  floatx4_t g_w2[4] = {}, g_w1 = {};
  float g_b2[4] = {}, g_w3[4] = {}, loss = 0.0f, g_b3 = 0.0f;
  const int64_t tiles = (nb + kTile - 1) / kTile;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    __syncthreads();  // parameters staged; the last tile's readers are done
    if (threadIdx.x < kTile * kInPad) {
      // features 0..5, then a row of ones (its products are the bias sums)
      const int k = threadIdx.x / kTile, c = threadIdx.x % kTile;
      const int64_t i = tile * kTile + c;
      float v = 0.0f;
      if (i < nb) {
        const int64_t at = idx ? static_cast<int64_t>(idx[i]) : i;
        v = k < kIn ? x[k * n + at] : (k == kIn ? 1.0f : 0.0f);
        if (k == 0) {
          s_t[c] = t[at];
          s_ok[c] = flag[at] == 0;
        }
      } else if (k == 0) {
        s_ok[c] = 0;  // no sample
      }
      s_x[k][c] = v;
    }
    __syncthreads();
    // H1: two steps of the 8 inputs (rows 6 and 7 of X are no inputs: W1's
    // padding columns are staged as zeros)
    floatx4_t h1 = {s_b1[row], s_b1[row + 1], s_b1[row + 2], s_b1[row + 3]};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = 2 * q + s;
      h1 = MfmaF32(s_w1[(16 * w + j) * 9 + k], s_x[k][j], h1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      h1[r] = Relu(h1[r]);
      s_h1[row + r][j] = h1[r];
    }
    __syncthreads();
    floatx4_t h2 = {s_b2[row], s_b2[row + 1], s_b2[row + 2], s_b2[row + 3]};
#pragma unroll
    for (int s = 0; s < 16; ++s)
      h2 = MfmaF32(s_w2[(16 * w + j) * kW2Stride + 16 * q + s], s_h1[16 * q + s][j], h2);
    float out = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      h2[r] = Relu(h2[r]);
      out += s_w3[row + r] * h2[r];
    }
    out += __shfl_xor(out, 16, 64);
    out += __shfl_xor(out, 32, 64);
    if (q == 0) s_y[w][j] = out;
    __syncthreads();
    if (threadIdx.x < kTile) {
      const float y = ((s_y[0][threadIdx.x] + s_y[1][threadIdx.x]) +
                       (s_y[2][threadIdx.x] + s_y[3][threadIdx.x])) + b3;
      const float e = s_ok[threadIdx.x] ? y - s_t[threadIdx.x] : 0.0f;
      const float ae = fabsf(e);
      const bool quad = !(huber > 0.0f) || ae <= huber;
      loss += (quad ? e * e : 2.0f * huber * ae - huber * huber) * inv_count;
      const float d = 2.0f * (quad ? e : copysignf(huber, e)) * inv_count;
      s_dy[threadIdx.x] = d;
      g_b3 += d;
    }
    __syncthreads();
    const float dy = s_dy[j];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float d2 = h2[r] > 0.0f ? dy * s_w3[row + r] : 0.0f;
      s_d2[row + r][j] = d2;
      g_b2[r] += d2;
      g_w3[r] += dy * h2[r];
    }
    __syncthreads();
    floatx4_t d1 = {};
#pragma unroll
    for (int s = 0; s < 16; ++s)
      d1 = MfmaF32(s_w2[(16 * q + s) * kW2Stride + 16 * w + j], s_d2[16 * q + s][j], d1);
#pragma unroll
    for (int r = 0; r < 4; ++r) s_d1[row + r][j] = h1[r] > 0.0f ? d1[r] : 0.0f;
    // sums over the tile's samples (index 4 s + q)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float a2 = s_d2[16 * w + j][4 * s + q];
#pragma unroll
      for (int m = 0; m < 4; ++m) g_w2[m] = MfmaF32(a2, s_h1[16 * m + j][4 * s + q], g_w2[m]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // this wave's own rows of dH1
#pragma unroll
    for (int s = 0; s < 4; ++s)
      g_w1 = MfmaF32(s_d1[16 * w + j][4 * s + q], s_x[j & 7][4 * s + q], g_w1);
  }
  float* out = part + static_cast<int64_t>(blockIdx.x) * kNParams;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (j < kInPad) {
      const float v = g_w1[r];
      out[kOffW1 + (row + r) * kInPad + j] = j < kIn ? v : 0.0f;
      if (j == kIn) out[kOffB1 + row + r] = v;
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) out[kOffW2 + (row + r) * kH + 16 * m + j] = g_w2[m][r];
    const float b2 = RowSum16(g_b2[r]), w3 = RowSum16(g_w3[r]);
    if (j == 0) {
      out[kOffB2 + row + r] = b2;
      out[kOffW3 + row + r] = w3;
    }
  }
  if (w == 0) {
    loss = RowSum16(loss);
    g_b3 = RowSum16(g_b3);
    if (lane == 0) {
      out[kOffB3] = g_b3;
      loss_part[blockIdx.x] = loss;
    }
  }
}

// Adam's update (p null: none).
struct AdamStep {
  float lr, b1, b2, eps, bc1, bc2;
  float *p, *m, *v;
};

// Sums the workgroups' partial gradients (and losses) in block order: 64
// parameters a workgroup, each wave a quarter of the blocks; writes grad
// (nullable) and the loss, and takes the Adam step (p nullable).
__global__ __launch_bounds__(kBlock) void MlpReduceKernel(const float* __restrict__ part,
                                                          const float* __restrict__ loss_part,
                                                          int nblocks, float* grad, float* loss,
                                                          AdamStep a) {
  __shared__ float s_g[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int k = blockIdx.x * 64 + lane;
  float g = 0.0f;
  if (k < kNParams) {
#pragma unroll 8
    for (int b = w; b < nblocks; b += 4) g += part[static_cast<int64_t>(b) * kNParams + k];
  }
  s_g[w][lane] = g;
  __syncthreads();
  if (w == 0 && k < kNParams) {
    g = (s_g[0][lane] + s_g[1][lane]) + (s_g[2][lane] + s_g[3][lane]);
    if (grad) grad[k] = g;
    // padding columns of W1 stay zero
    if (a.p && !(k < kOffB1 && (k % kInPad) >= kIn)) {
      const float m = a.b1 * a.m[k] + (1.0f - a.b1) * g;
      const float v = a.b2 * a.v[k] + (1.0f - a.b2) * g * g;
      a.m[k] = m;
      a.v[k] = v;
      const float mh = m / a.bc1, vh = v / a.bc2;
      a.p[k] -= a.lr * mh / (sqrtf(vh) + a.eps);
    }
  }
  if (blockIdx.x == 0 && w == 1) {
    float l = 0.0f;
    for (int b = lane; b < nblocks; b += 64) l += loss_part[b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off, 64);
    if (lane == 0) *loss = l;
  }
}

} // namespace
} // namespace fvs

// ---- host side -----------------------------------------------------------------

using namespace fvs;

struct fvs_mlp {
  hipStream_t stream;
  float* params;  // FP32 master (device)
  float* adam_m;
  float* adam_v;
  float* grad;
  float* loss;
  short* tiles;   // packed bf16 A operands
  float* bias;    // b1, b2, b3
  int64_t adam_t;
  // dataset
  int64_t n;
  double* prim;
  float* x;
  float* target;
  int* flag;
  int* iters;
  float* part;       // partial gradients, kGradBlocks x kNParams
  float* loss_part;  // kGradBlocks
};

namespace {

int Alloc(void** p, size_t bytes) {
  if (hipMalloc(p, bytes) != hipSuccess) {
    SetError("hipMalloc of %zu bytes failed", bytes);
    return FVS_HIP_ERROR;
  }
  return FVS_OK;
}

int Pack(fvs_mlp* m) {
  hipLaunchKernelGGL(MlpPackKernel, dim3(kNTiles), dim3(64), 0, m->stream, m->params, m->tiles,
                     m->bias);
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

// Partial gradients of a batch (idx nullable: samples 0 .. nb - 1) and their
// reduction.  grad (nullable) and loss: device memory.
int BatchGradients(fvs_mlp* m, const float* x, const float* t, const int* flag, int64_t n,
                   const uint32_t* idx, int64_t nb, float inv_count, float huber, float* grad,
                   float* loss, const AdamStep& adam) {
  const int64_t tiles = (nb + kTile - 1) / kTile;
  const int blocks = static_cast<int>(tiles < kGradBlocks ? tiles : kGradBlocks);
  hipLaunchKernelGGL(MlpGradKernel, dim3(blocks), dim3(kBlock), 0, m->stream, m->params, x, t,
                     flag, n, idx, nb, inv_count, huber, m->part, m->loss_part);
  FVS_LAUNCH_CHECK();
  hipLaunchKernelGGL(MlpReduceKernel, dim3((kNParams + 63) / 64), dim3(kBlock), 0, m->stream,
                     m->part, m->loss_part, blocks, grad, loss, adam);
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

uint64_t HostSplitMix(uint64_t& s) {
  s += 0x9E3779B97F4A7C15ull;
  uint64_t z = s;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

} // namespace

// Initial guesses for every face of direction dir of a ghost-free
// transmissive patch (face box n with n[dir] + 1, x fastest), on stream s.
void fvs::MlpOperands(const fvs_mlp* m, const short** tiles, const float** bias) {
  *tiles = m->tiles;
  *bias = m->bias;
}

int fvs::MlpFaceGuess(fvs_mlp* m, hipStream_t s, int dim, double gamma,
                      const double* const* cons, const int64_t n[3], int dir, double* guess) {
  if (!m || !cons || !n || !guess || (dim != 2 && dim != 3) || dir < 0 || dir >= dim) {
    SetError("bad argument");
    return FVS_BAD_ARGUMENT;
  }
  const int64_t nx = n[0], ny = n[1], nz = dim == 3 ? n[2] : 1;
  const int64_t nf = (nx + (dir == 0)) * (ny + (dir == 1)) * (nz + (dir == 2));
  const unsigned blocks = unsigned((nf + kBlock - 1) / kBlock);
  const double gm1inv = 1.0 / (gamma - 1.0);
  const double* u4 = dim == 3 ? cons[4] : nullptr;
#define FVS_MIF(DD, DR)                                                                          \
  hipLaunchKernelGGL((MlpInferFaces<DD, DR>), dim3(blocks), dim3(kBlock), 0, s, cons[0],         \
                     cons[1], cons[2], cons[3], u4, nx, ny, nz, gamma, gm1inv, m->tiles, m->bias,  \
                     guess)
  if (dim == 2) {
    if (dir == 0) FVS_MIF(2, 0); else FVS_MIF(2, 1);
  } else {
    if (dir == 0) FVS_MIF(3, 0); else if (dir == 1) FVS_MIF(3, 1); else FVS_MIF(3, 2);
  }
#undef FVS_MIF
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

extern "C" {

int fvs_mlp_create(void* hip_stream, uint64_t seed, fvs_mlp** out) {
  if (!out) {
    SetError("null output pointer");
    return FVS_BAD_ARGUMENT;
  }
  *out = nullptr;
  fvs_mlp* m = new (std::nothrow) fvs_mlp();
  if (!m) {
    SetError("out of host memory");
    return FVS_BAD_ARGUMENT;
  }
  std::memset(m, 0, sizeof *m);
  m->stream = static_cast<hipStream_t>(hip_stream);
  const size_t pb = kNParams * sizeof(float);
  if (Alloc((void**)&m->params, pb) || Alloc((void**)&m->adam_m, pb) ||
      Alloc((void**)&m->adam_v, pb) || Alloc((void**)&m->grad, pb) ||
      Alloc((void**)&m->loss, sizeof(float)) ||
      Alloc((void**)&m->part, kGradBlocks * pb) ||
      Alloc((void**)&m->loss_part, kGradBlocks * sizeof(float)) ||
      Alloc((void**)&m->tiles, kNTiles * kTileShorts * sizeof(short)) ||
      Alloc((void**)&m->bias, (2 * kH + 1) * sizeof(float))) {
    delete m;
    return FVS_HIP_ERROR;
  }
  // He-uniform initialisation of the ReLU layers (Glorot for the linear
  // output) from SplitMix64, zero biases and padding.
  std::vector<float> p(kNParams, 0.0f);
  uint64_t st = seed;
  auto uni = [&](float a) {
    return static_cast<float>((HostSplitMix(st) >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0) * a;
  };
  const float a1 = std::sqrt(6.0f / kIn), a2 = std::sqrt(6.0f / kH),
              a3 = std::sqrt(6.0f / (kH + 1));
  for (int o = 0; o < kH; ++o)
    for (int k = 0; k < kIn; ++k) p[kOffW1 + o * kInPad + k] = uni(a1);
  for (int k = 0; k < kH * kH; ++k) p[kOffW2 + k] = uni(a2);
  for (int k = 0; k < kH; ++k) p[kOffW3 + k] = uni(a3);
  FVS_HIP_CHECK(hipMemcpyAsync(m->params, p.data(), pb, hipMemcpyHostToDevice, m->stream));
  FVS_HIP_CHECK(hipMemsetAsync(m->adam_m, 0, pb, m->stream));
  FVS_HIP_CHECK(hipMemsetAsync(m->adam_v, 0, pb, m->stream));
  if (int rc = Pack(m)) return rc;
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  *out = m;
  return FVS_OK;
}

int fvs_mlp_destroy(fvs_mlp* m) {
  if (!m) return FVS_OK;
  (void)hipStreamSynchronize(m->stream);
  void* ps[] = {m->params, m->adam_m, m->adam_v, m->grad, m->loss, m->tiles, m->bias,
                m->part, m->loss_part,
                m->prim, m->x, m->target, m->flag, m->iters};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  delete m;
  return FVS_OK;
}

int fvs_mlp_num_params(void) { return kNParams; }

int fvs_mlp_get_params(fvs_mlp* m, float* host) {
  if (!m || !host) {
    SetError("null argument");
    return FVS_BAD_ARGUMENT;
  }
  FVS_HIP_CHECK(hipMemcpyAsync(host, m->params, kNParams * sizeof(float), hipMemcpyDeviceToHost,
                               m->stream));
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  return FVS_OK;
}

int fvs_mlp_set_params(fvs_mlp* m, const float* host) {
  if (!m || !host) {
    SetError("null argument");
    return FVS_BAD_ARGUMENT;
  }
  FVS_HIP_CHECK(hipMemcpyAsync(m->params, host, kNParams * sizeof(float), hipMemcpyHostToDevice,
                               m->stream));
  if (int rc = Pack(m)) return rc;
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  return FVS_OK;
}

int fvs_mlp_generate(fvs_mlp* m, int64_t n, uint64_t seed, double gamma, int64_t counts[3]) {
  if (!m || n <= 0) {
    SetError("bad argument");
    return FVS_BAD_ARGUMENT;
  }
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  void* ps[] = {m->prim, m->x, m->target, m->flag, m->iters};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  m->prim = nullptr;
  m->x = m->target = nullptr;
  m->flag = m->iters = nullptr;
  if (Alloc((void**)&m->prim, n * 6 * sizeof(double)) ||
      Alloc((void**)&m->x, n * kIn * sizeof(float)) ||
      Alloc((void**)&m->target, n * sizeof(float)) || Alloc((void**)&m->flag, n * sizeof(int)) ||
      Alloc((void**)&m->iters, n * sizeof(int)))
    return FVS_HIP_ERROR;
  m->n = n;
  hipLaunchKernelGGL(MlpSampleKernel, dim3(unsigned((n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     m->stream, n, seed, gamma, 5000, 1e-7, m->prim, m->x, m->target, m->flag,
                     m->iters);
  FVS_LAUNCH_CHECK();
  if (counts) {
    std::vector<int> f(n);
    FVS_HIP_CHECK(hipMemcpyAsync(f.data(), m->flag, n * sizeof(int), hipMemcpyDeviceToHost,
                                 m->stream));
    FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
    counts[0] = counts[1] = counts[2] = 0;
    for (int64_t i = 0; i < n; ++i) counts[f[i] < 3 ? f[i] : 2] += 1;
  }
  return FVS_OK;
}

// Copies the generated dataset into caller device buffers (each nullable;
// all null just reports n).
int fvs_mlp_dataset(fvs_mlp* m, int64_t* n, double* prim, float* x, float* target, int* flag,
                    int* iters) {
  if (!m) {
    SetError("null mlp");
    return FVS_BAD_ARGUMENT;
  }
  if (n) *n = m->n;
  if ((prim || x || target || flag || iters) && !m->prim) {
    SetError("no dataset generated");
    return FVS_BAD_ARGUMENT;
  }
  const int64_t k = m->n;
  const hipMemcpyKind d2d = hipMemcpyDeviceToDevice;
  if (prim) FVS_HIP_CHECK(hipMemcpyAsync(prim, m->prim, k * 6 * sizeof(double), d2d, m->stream));
  if (x) FVS_HIP_CHECK(hipMemcpyAsync(x, m->x, k * kIn * sizeof(float), d2d, m->stream));
  if (target) FVS_HIP_CHECK(hipMemcpyAsync(target, m->target, k * sizeof(float), d2d, m->stream));
  if (flag) FVS_HIP_CHECK(hipMemcpyAsync(flag, m->flag, k * sizeof(int), d2d, m->stream));
  if (iters) FVS_HIP_CHECK(hipMemcpyAsync(iters, m->iters, k * sizeof(int), d2d, m->stream));
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  return FVS_OK;
}

// FP32 forward of n samples (x: 6 x n device floats) -> y (device floats).
int fvs_mlp_forward(fvs_mlp* m, const float* x, int64_t n, float* y) {
  if (!m || !x || !y || n <= 0) {
    SetError("bad argument");
    return FVS_BAD_ARGUMENT;
  }
  hipLaunchKernelGGL(MlpForwardKernel, dim3(unsigned((n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     m->stream, m->params, x, n, y);
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

// Loss (mean over samples with flag 0 of e^2, or of the Huber form when
// huber > 0) and its gradient on one batch (device arrays x: 6 x n,
// target: n, flag: n); grad_host gets the kNParams gradient.
int fvs_mlp_gradients(fvs_mlp* m, const float* x, const float* target, const int* flag,
                      int64_t n, float huber, float* grad_host, float* loss_host) {
  if (!m || !x || !target || !flag || n <= 0) {
    SetError("bad argument");
    return FVS_BAD_ARGUMENT;
  }
  std::vector<int> f(n);
  FVS_HIP_CHECK(hipMemcpyAsync(f.data(), flag, n * sizeof(int), hipMemcpyDeviceToHost, m->stream));
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  int64_t valid = 0;
  for (int64_t i = 0; i < n; ++i) valid += (f[i] == 0);
  if (int rc = BatchGradients(m, x, target, flag, n, nullptr, n,
                              valid > 0 ? 1.0f / float(valid) : 0.0f, huber, m->grad, m->loss,
                              AdamStep{}))
    return rc;
  if (grad_host)
    FVS_HIP_CHECK(hipMemcpyAsync(grad_host, m->grad, kNParams * sizeof(float),
                                 hipMemcpyDeviceToHost, m->stream));
  if (loss_host)
    FVS_HIP_CHECK(hipMemcpyAsync(loss_host, m->loss, sizeof(float), hipMemcpyDeviceToHost, m->stream));
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  return FVS_OK;
}

// Adam training on the generated dataset: `epochs` passes in minibatches of
// `batch` samples (deterministic shuffles from `seed`), learning rate
// lr * (1 + cos(pi t / T)) / 2 over the T steps of the call, Huber loss
// with threshold `huber` (0: squared error).  loss_history (host, nullable)
// receives a smoothed minibatch loss per epoch.
int fvs_mlp_train(fvs_mlp* m, int epochs, int64_t batch, float lr, float huber, uint64_t seed,
                  float* loss_history) {
  if (!m || !m->x || epochs < 0 || batch <= 0) {
    SetError("bad argument (dataset generated?)");
    return FVS_BAD_ARGUMENT;
  }
  const int64_t n = m->n;
  std::vector<int> flags(n);
  FVS_HIP_CHECK(hipMemcpyAsync(flags.data(), m->flag, n * sizeof(int), hipMemcpyDeviceToHost,
                               m->stream));
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  // Sample indices fit 32 bits: 2^32 samples (84 bytes each) exceed the card.
  std::vector<uint32_t> valid;
  valid.reserve(n);
  for (int64_t i = 0; i < n; ++i)
    if (flags[i] == 0) valid.push_back(static_cast<uint32_t>(i));
  const int64_t nv = static_cast<int64_t>(valid.size());
  if (nv < batch) {
    SetError("dataset has %lld valid samples, fewer than one batch", (long long)nv);
    return FVS_BAD_ARGUMENT;
  }
  const int64_t nbatches = nv / batch;
  // Device: two epochs' permutations (the next one is shuffled and uploaded
  // while an epoch runs) and their steps' losses; host: pinned staging of both.
  // A single epoch stages in pageable memory.
  uint32_t* perm = nullptr;
  float* losses = nullptr;
  char* stage = nullptr;
  hipEvent_t done[2] = {nullptr, nullptr};  // an epoch's steps and loss copy
  const size_t pbytes = nv * sizeof(uint32_t), lbytes = nbatches * sizeof(float);
  const int nbuf = epochs > 1 ? 2 : 1;
  std::vector<float> one(nbuf == 1 ? nbatches : 0);
  int rc = FVS_OK;
  if (Alloc((void**)&perm, nbuf * pbytes) || Alloc((void**)&losses, nbuf * lbytes))
    rc = FVS_HIP_ERROR;
  if (rc == FVS_OK && nbuf > 1) {
    if (hipHostMalloc(&stage, nbuf * (pbytes + lbytes), hipHostMallocDefault) != hipSuccess ||
        hipEventCreateWithFlags(&done[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&done[1], hipEventDisableTiming) != hipSuccess) {
      SetError("training buffers failed");
      rc = FVS_HIP_ERROR;
    }
  }
  float* host_losses = stage ? reinterpret_cast<float*>(stage + nbuf * pbytes) : one.data();
  // The smoothed loss of epoch e, whose losses have arrived.
  auto record = [&](int e) {
    const float* l = host_losses + (e % nbuf) * nbatches;
    double smooth = 0.0;
    for (int64_t b = 0; b < nbatches; ++b) {
      if (b % 64 != 0 && b != nbatches - 1) continue;
      smooth = (b == 0) ? l[b] : 0.9 * smooth + 0.1 * l[b];
    }
    loss_history[e] = static_cast<float>(smooth);
  };
  uint64_t st = seed;
  AdamStep adam{};
  adam.b1 = 0.9f;
  adam.b2 = 0.999f;
  adam.eps = 1e-8f;
  adam.p = m->params;
  adam.m = m->adam_m;
  adam.v = m->adam_v;
  const double total = static_cast<double>(epochs) * static_cast<double>(nbatches);
  int64_t step = 0;
  for (int e = 0; e < epochs && rc == FVS_OK; ++e) {
    for (int64_t i = nv - 1; i > 0; --i) {
      const int64_t j = static_cast<int64_t>(HostSplitMix(st) % static_cast<uint64_t>(i + 1));
      std::swap(valid[i], valid[j]);
    }
    const int buf = e % nbuf;
    uint32_t* dst = perm + buf * nv;
    const void* src = valid.data();
    if (stage) {
      // the epoch before last has left its buffers
      if (e >= 2) {
        if (hipEventSynchronize(done[buf]) != hipSuccess) rc = FVS_HIP_ERROR;
        if (rc == FVS_OK && loss_history) record(e - 2);
      }
      src = std::memcpy(stage + buf * pbytes, valid.data(), pbytes);
    }
    if (rc != FVS_OK ||
        hipMemcpyAsync(dst, src, pbytes, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
        (!stage && hipStreamSynchronize(m->stream) != hipSuccess)) {
      SetError("permutation upload failed");
      rc = FVS_HIP_ERROR;
      break;
    }
    for (int64_t b = 0; b < nbatches && rc == FVS_OK; ++b) {
      m->adam_t += 1;
      step += 1;
      adam.bc1 = 1.0f - std::pow(adam.b1, float(m->adam_t));
      adam.bc2 = 1.0f - std::pow(adam.b2, float(m->adam_t));
      adam.lr =
          static_cast<float>(lr * 0.5 * (1.0 + std::cos(3.141592653589793 * step / total)));
      rc = BatchGradients(m, m->x, m->target, m->flag, n, dst + b * batch, batch,
                          1.0f / float(batch), huber, nullptr, losses + buf * nbatches + b, adam);
    }
    if (rc != FVS_OK) break;
    if ((loss_history &&
         hipMemcpyAsync(host_losses + buf * nbatches, losses + buf * nbatches, lbytes,
                        hipMemcpyDeviceToHost, m->stream) != hipSuccess) ||
        (stage && hipEventRecord(done[buf], m->stream) != hipSuccess)) {
      SetError("loss readback failed");
      rc = FVS_HIP_ERROR;
    }
  }
  if (hipStreamSynchronize(m->stream) != hipSuccess && rc == FVS_OK) {
    SetError("training failed");
    rc = FVS_HIP_ERROR;
  }
  if (rc == FVS_OK && loss_history)
    for (int e = std::max(0, epochs - nbuf); e < epochs; ++e) record(e);
  if (perm) (void)hipFree(perm);
  if (losses) (void)hipFree(losses);
  if (stage) (void)hipHostFree(stage);
  for (hipEvent_t ev : done)
    if (ev) (void)hipEventDestroy(ev);
  if (rc != FVS_OK) return rc;
  if (int rc = Pack(m)) return rc;
  FVS_HIP_CHECK(hipStreamSynchronize(m->stream));
  return FVS_OK;
}

// Matrix-core (BF16 MFMA) inference on complete state pairs.
int fvs_mlp_infer_pairs(fvs_mlp* m, int dim, int dir, const double* left, const double* right,
                        int64_t n, float* r_out, double* guess) {
  if (!m || !left || !right || n <= 0 || (dim != 2 && dim != 3) || dir < 0 || dir >= dim) {
    SetError("bad argument");
    return FVS_BAD_ARGUMENT;
  }
  const unsigned blocks = unsigned((n + kBlock - 1) / kBlock);
  if (dim == 2)
    hipLaunchKernelGGL(MlpInferPairs<2>, dim3(blocks), dim3(kBlock), 0, m->stream, left, right, n,
                       dir, m->tiles, m->bias, r_out, guess);
  else
    hipLaunchKernelGGL(MlpInferPairs<3>, dim3(blocks), dim3(kBlock), 0, m->stream, left, right, n,
                       dir, m->tiles, m->bias, r_out, guess);
  FVS_LAUNCH_CHECK();
  return FVS_OK;
}

int fvs_mlp_face_guess(fvs_mlp* m, int dim, double gamma, const double* const* cons,
                       const int64_t n[3], int dir, double* guess) {
  if (!m) {
    SetError("null mlp");
    return FVS_BAD_ARGUMENT;
  }
  return MlpFaceGuess(m, m->stream, dim, gamma, cons, n, dir, guess);
}

} // extern "C"
