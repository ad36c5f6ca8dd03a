// Learned Newton initial guess for the Noble 2D inversion.
//
// A multilayer perceptron 8 -> 64 -> 64 -> 1 (tanh) maps dimensionless
// invariants of the conserved state, the metric and the plain guess to the
// correction log(W / W_guess), W being the enthalpy-like unknown of the 2D
// scheme and W_guess the reference's start (from the previous primitives).
// Weights live in FP32 (training) with BF16 copies for the matrix cores: the
// two hidden layers run on gfx950 MFMA (v_mfma_f32_16x16x32_bf16, FP32
// accumulate), 16 inversions per tile.
//
//   k_mlp_features  FP64 set-up of the inversion -> 8 features per zone, and
//                   the training target log(W_solved / W_guess)
//   k_mlp_forward   features -> prediction (MFMA; each wavefront keeps the
//                   network in registers and runs over 16-sample tiles)
//   k_mlp_backward  forward + backward of 16-sample tiles on the matrix cores
//                   (FP64, with the BF16 roundings of the inference), a partial
//                   sum of every weight's gradient per block
//   k_mlp_update    the partial sums added up, Adam, the BF16 copies of the
//                   hidden-layer weights (or the gradient alone)
//   k_mlp_set       the parameters a caller sets, the copies, the zeros of a gradient
//   k_c2p_learned   the mixed-precision inversion (FP32 Newton, polish,
//                   double-double primitives) from the learned start where
//                   the network predicts a large correction and the start's
//                   first FP64 Newton step passes a size check, else from
//                   the plain start; a zone that does not converge joins
//                   the list that the reference path (HG_C2P_REFINED)
//                   inverts from the plain guess
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "harmgpu.h"
#include "hg_c2p.h"
#include "hg_c2p_io.h"
#include "hg_host.h"

using namespace hg;

namespace {

constexpr int NIN = 8, NH = 64;
// parameter block (FP32): W1[8][64] b1[64] W2[64][64] b2[64] W3[64] b3 mu[8] sd[8]
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + NIN * NH, OFF_W2 = OFF_B1 + NH, OFF_B2 = OFF_W2 + NH * NH,
              OFF_W3 = OFF_B2 + NH, OFF_B3 = OFF_W3 + NH, OFF_MU = OFF_B3 + 1, OFF_SD = OFF_MU + NIN,
              NPARAM = OFF_SD + NIN;
// trainable parameters are [0, OFF_MU)
constexpr int NTRAIN = OFF_MU;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// W = (rho + gam u) (1 + u~^2) of primitives p
__device__ __forceinline__ double W_of_prims(const Geom &G, const double *p, double gam) {
  double utsq = 0.;
#pragma unroll
  for (int i = 1; i < 4; i++)
#pragma unroll
    for (int j = 1; j < 4; j++) utsq += G.gcov[i][j] * p[U1 + i - 1] * p[U1 + j - 1];
  return (p[RHO] + gam * p[UU]) * (1.0 + utsq);
}

// features X[n][8] from the plain guess; with solved primitives, the
// training target y = log(W_solved / W_guess) in FP64 rounded once to FP32
__global__ void __launch_bounds__(256) k_mlp_features(int64_t n, double gam, const double *__restrict__ U,
                                                      const double *__restrict__ gcov,
                                                      const double *__restrict__ gcon,
                                                      const double *__restrict__ gdet,
                                                      const double *__restrict__ guess,
                                                      const double *__restrict__ solved, float *__restrict__ X,
                                                      float *__restrict__ y, int *__restrict__ ok) {
  int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n) return;
  Geom G;
  double u[NPR], p[NPR], Ug[NPR];
  load_batch_zone(n, t, U, gcov, gcon, gdet, guess, G, u, p);
  C2PInv c;
  double W_last, alpha;
  int code = c2p_setup_zone(u, G, gam, p, c, W_last, alpha, Ug);
  float x[NIN];
  c2p_features(c, W_last, alpha, gam, x);
  bool good = (code == 0);
#pragma unroll
  for (int k = 0; k < NIN; k++) {
    good = good && isfinite(x[k]);
    X[t * NIN + k] = x[k];
  }
  if (solved) {
    double ps[NPR];
#pragma unroll
    for (int pl = 0; pl < NPR; pl++) ps[pl] = solved[pl * n + t];
    double yt = log(W_of_prims(G, ps, gam) / W_last);
    good = good && isfinite(yt);
    if (y) y[t] = (float)yt;
  }
  if (ok) ok[t] = good ? 1 : 0;
}

// ---------------------------------------------------------------------------
// forward pass on the matrix cores: one wavefront, 16 samples per MFMA tile.
// v_mfma_f32_16x16x32_bf16 lane layout (lane l, q = l / 16, r = l % 16):
//   A (16 x 32):  A[r][8q + j], j = 0..7
//   B (32 x 16):  B[8q + j][r]
//   C (16 x 16):  C[4q + i][r], i = 0..3
// The network input x enters as a pair of BF16 numbers hi = bf16(x),
// lo = bf16(x - hi) against the same BF16 weights in both halves of K, so
// the product keeps ~16 bits of the input (the weights are BF16, the
// accumulation FP32): layer 1 has K = 32 = [x_hi(8) x_lo(8) 0(16)].  The
// hidden activations enter layer 2 as BF16 (K = 64).
// ---------------------------------------------------------------------------
struct MlpDev {
  float *w;       // FP32 parameters (biases, W3, normalisation)
  __bf16 *w1b;    // BF16 W1 B-fragments: [nt 4][lane 64][j 8] of the K = 32 layer-1 matrix
  __bf16 *w2b;    // BF16 W2 B-fragments: [ks 2][nt 4][lane 64][j 8]
  float *w2q;     // the BF16 W2 in FP32, [64][64]
  float *wlo;     // what the FP32 parameters round off of the trained ones
};

// the network as one wavefront holds it: the B-fragments of both hidden
// layers (lane l = 16 q + r holds rows 8 q .. 8 q + 7 of column 16 nt + r),
// and the biases and output weights of the lane's columns 16 nt + r
struct MlpRegs {
  bf16x8 w1[4], w2[8];
  float b1[4], b2[4], w3[4], b3;
};

__device__ __forceinline__ void mlp_load(const MlpDev &m, MlpRegs &R) {
  const int l = threadIdx.x & 63, r = l & 15;
#pragma unroll
  for (int nt = 0; nt < 4; nt++) {
    R.w1[nt] = *(const bf16x8 *)(m.w1b + (nt * 64 + l) * 8);
    R.b1[nt] = m.w[OFF_B1 + 16 * nt + r];
    R.b2[nt] = m.w[OFF_B2 + 16 * nt + r];
    R.w3[nt] = m.w[OFF_W3 + 16 * nt + r];
  }
#pragma unroll
  for (int f = 0; f < 8; f++) R.w2[f] = *(const bf16x8 *)(m.w2b + (f * 64 + l) * 8);
  R.b3 = m.w[OFF_B3];
}

__device__ __forceinline__ __bf16 bf_hi(float v) { return (__bf16)v; }

// tanh as 1 - 2 / (exp(2x) + 1) with the hardware exponential (of base 2) and
// reciprocal (absolute error ~1e-7; saturates to +-1 without overflow).  The
// factors 2 are exact, so they ride on the product and the last subtraction:
// five instructions instead of seven, k_c2p_learned 163 -> 155 us
__device__ __forceinline__ float act(float x) {
  const float e = __builtin_amdgcn_exp2f(x * 0x1.715476p+1f);  // 2 log2(e)
  return fmaf(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f);
}
__device__ __forceinline__ __bf16 bf_lo(float v) { return (__bf16)(v - (float)(__bf16)v); }

// rows of forward16's scratch in LDS: four floats apart in the banks, so the 16
// lanes of a column block read 16 rows as 16-byte vectors without conflicts
constexpr int NHS = NH + 4;

// 16 samples: xin[16][8] (normalised) -> y[16]; h[16][NHS] float LDS scratch
// for the layer-1 activations (the C layout of layer 1 -- sample 4 q + i in
// lane 16 q + r -- is not the A layout of layer 2, sample r in lane 16 q + r);
// layer 3 is summed per lane over its columns, then across the 16 lanes of
// each sample group
__device__ __forceinline__ void forward16(const MlpRegs &R, const float (*xin)[NIN], float (*h)[NHS], float *y) {
  const int l = threadIdx.x & 63, q = l >> 4, r = l & 15;
  // layer 1
  bf16x8 a;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    float v = (q < 2) ? xin[r][j] : 0.0f;
    a[j] = (q == 0) ? bf_hi(v) : bf_lo(v);  // q >= 2: bf16(0 - 0) = 0
  }
#pragma unroll
  for (int nt = 0; nt < 4; nt++) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, R.w1[nt], acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) h[4 * q + i][16 * nt + r] = act(acc[i] + R.b1[nt]);
  }
  __syncthreads();
  // layer 2: K = 64 in two steps, BF16 inputs
  f32x4 acc2[4];
#pragma unroll
  for (int nt = 0; nt < 4; nt++) acc2[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    const int kb = 32 * ks + 8 * q;
    bf16x8 a2;
#pragma unroll
    for (int j = 0; j < 8; j++) a2[j] = bf_hi(h[r][kb + j]);
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
      acc2[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, R.w2[4 * ks + nt], acc2[nt], 0, 0, 0);
  }
  // layer 3: lane (q, r) sums its four columns for samples 4 q + i
  float part[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float sacc = 0.f;
#pragma unroll
    for (int nt = 0; nt < 4; nt++) sacc += act(acc2[nt][i] + R.b2[nt]) * R.w3[nt];
    part[i] = sacc;
  }
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1)
#pragma unroll
    for (int i = 0; i < 4; i++) part[i] += __shfl_xor(part[i], off, 64);
  if (r == 0)
#pragma unroll
    for (int i = 0; i < 4; i++) y[4 * q + i] = R.b3 + part[i];
  __syncthreads();
}

// one wavefront per block holds the network in registers and runs over
// tiles of 16 samples (grid-stride)
__device__ __forceinline__ void mlp_forward_body(int64_t n, const float *__restrict__ X, float *__restrict__ y,
                                                 const MlpDev &m, unsigned bid, unsigned nblk) {
  __shared__ float xin[16][NIN];
  __shared__ __align__(16) float h[16][NHS];
  __shared__ float yo[16];
  const int l = threadIdx.x;
  MlpRegs R;
  mlp_load(m, R);
  // lane 8 s + k (s < 8) normalises feature k of sample s and of s + 8
  const int k = l & 7;
  const float mk = m.w[OFF_MU + k], sk = m.w[OFF_SD + k];
  for (int64_t base = (int64_t)bid * 16; base < n; base += (int64_t)nblk * 16) {
#pragma unroll
    for (int half = 0; half < 2; half++) {
      const int s = half * 8 + (l >> 3);
      const int64_t t = base + s;
      xin[s][k] = (t < n) ? (X[t * NIN + k] - mk) / sk : 0.f;
    }
    __syncthreads();
    forward16(R, xin, h, yo);
    if (l < 16 && base + l < n) y[base + l] = yo[l];
    __syncthreads();
  }
}

__global__ void __launch_bounds__(64) k_mlp_forward(int64_t n, const float *__restrict__ X, float *__restrict__ y,
                                                    MlpDev m) {
  mlp_forward_body(n, X, y, m, blockIdx.x, gridDim.x);
}

// grouped: every grid's step features through the one network
__global__ void __launch_bounds__(64) kg_mlp_forward(const GridView *__restrict__ views,
                                                     const unsigned *__restrict__ first, int ng, MlpDev m) {
  const int g_ = group_of(first, ng, blockIdx.x);
  const GridView &v = views[g_];
  const int64_t n = (int64_t)v.d.n1 * v.d.n2 * v.d.n3;
  mlp_forward_body(n, v.lx, v.ly, m, blockIdx.x - first[g_], first[g_ + 1] - first[g_]);
}

// BF16 copies of hidden-layer weight e (its value in w1b / w2b at every place
// of the B-fragments: layer 1 [nt][l][j] = W1x[8 q + j][16 nt + r], lane
// l = 16 q + r, with W1x the K = 32 matrix whose rows 0..7 and 8..15 are both
// W1, the input's hi and lo halves, and whose rows 16..31 stay zero; layer 2
// [ks][nt][l][j] = W2[32 ks + 8 q + j][16 nt + r]) and, for the backward pass,
// the rounded W2 in FP32
__device__ __forceinline__ void refresh_bf16(int e, float v, const MlpDev &m) {
  if (e < OFF_B1) {
    const int i = e / NH, c = e % NH, nt = c >> 4, r = c & 15;
    m.w1b[(nt * 64 + r) * 8 + i] = (__bf16)v;
    m.w1b[(nt * 64 + 16 + r) * 8 + i] = (__bf16)v;
  } else if (e >= OFF_W2 && e < OFF_B2) {
    const int k = (e - OFF_W2) / NH, c = (e - OFF_W2) % NH, nt = c >> 4, r = c & 15;
    const int ks = k >> 5, q = (k >> 3) & 3, j = k & 7;
    m.w2b[((ks * 4 + nt) * 64 + 16 * q + r) * 8 + j] = (__bf16)v;
    m.w2q[e - OFF_W2] = (float)(__bf16)v;
  }
}

// ---------------------------------------------------------------------------
// backward pass: a block of four wavefronts runs over tiles of 16 samples, and
// wavefront w has columns 16 w .. 16 w + 15 of every layer.  The forward is
// recomputed with the BF16-rounded weights and layer inputs of the inference
// (hi + lo input, BF16 hidden activations; the roundings are treated as the
// identity when differentiating: the gradient is that of the master weights),
// and all arithmetic is FP64 on v_mfma_f64_16x16x4_f64:
//   z2 = h1 W2, dz1 = (dz2 W2^T) (1 - h1^2), dW2 = h1^T dz2, dW1 = x^T dz1
// A hidden activation or weight then rounds to the BF16 number of the exact
// computation, where FP32 sums land on the other side now and then and Adam
// carries that on: two epochs of 128 minibatches end 1.7e-8 from 64-bit
// training (the parameters' own FP32 rounding), in FP32 4e-4.  It costs 3 us a
// minibatch of 2048, the block being bound by its launch and a few memory
// latencies more than by its products.  A C-layout result (sample 4 i + q in lane 16 q + r, register i) is at
// once a B operand of a product summed over the samples: step i takes sample
// 4 i + q in slot q, and A is read from LDS in that order.  The gradients stay
// in accumulators over the block's tiles and go out once per block, to a row
// of partial sums of its own: sums in a fixed order, no atomics.
// A minibatch of 2048 is 128 one-tile blocks.  One wavefront per 64 samples on
// the vector units with an atomic per weight and block took 136 us (32 of them
// on 1024 SIMDs), Adam and the copies two more launches of 4.7 us; now 11.6 us
// here and 3.9 in k_mlp_update.
// ---------------------------------------------------------------------------
typedef double f64x4 __attribute__((ext_vector_type(4)));

// the value a layer input carries into the matrix cores: hi + lo
__device__ __forceinline__ double eff(double v) {
  const float hi = (float)bf_hi((float)v);
  return (double)hi + (double)(float)bf_hi((float)(v - (double)hi));
}
__device__ __forceinline__ double act64(double x) { return 1.0 - 2.0 / (exp(2.0 * x) + 1.0); }

constexpr int BACK_BLOCKS = 256;                   // most partial sums
constexpr int PART = (NTRAIN + 1 + 63) / 64 * 64;  // their stride: the weights, then the loss

__global__ void __launch_bounds__(256) k_mlp_backward(int64_t n, const float *__restrict__ X,
                                                      const float *__restrict__ Y, MlpDev m, double inv_n,
                                                      double loss_scale, double *__restrict__ part) {
  __shared__ double xs[16][NIN], dz2s[16][NH + 1], ys[4][16];
  __shared__ float h1q[16][NH + 4];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, q = l >> 4, r = l & 15;
  const int col = 16 * w + r;
  // thread 8 s + k (of the first 128) has feature k of sample s; a tile's
  // samples are on their way while the weights, or the tile before, are
  const int xs_s = threadIdx.x / NIN, xs_k = threadIdx.x % NIN;
  float nx = 0.f, ny[4] = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int64_t b) {
    if (xs_s < 16) nx = b + xs_s < n ? X[(b + xs_s) * NIN + xs_k] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) ny[i] = b + 4 * i + q < n ? Y[b + 4 * i + q] : 0.f;
  };
  fetch((int64_t)blockIdx.x * 16);
  const double mu = m.w[OFF_MU + xs_k], sd = m.w[OFF_SD + xs_k];
  const bf16x8 w1 = *(const bf16x8 *)(m.w1b + (w * 64 + r) * 8);  // rows 0..7 of column col
  float w2[16], w2t[16];  // W2 and W2^T as B operands: elements (4 step + q, col)
#pragma unroll
  for (int st = 0; st < 16; st++) {
    w2[st] = m.w2q[(4 * st + q) * NH + col];
    w2t[st] = m.w2q[col * NH + 4 * st + q];
  }
  auto par = [&](int e) { return (double)m.w[e] + (double)m.wlo[e]; };
  const double b1 = par(OFF_B1 + col), b2 = par(OFF_B2 + col), w3 = par(OFF_W3 + col), b3 = par(OFF_B3);
  f64x4 gW2[4], gW1 = {0., 0., 0., 0.};
#pragma unroll
  for (int kt = 0; kt < 4; kt++) gW2[kt] = (f64x4){0., 0., 0., 0.};
  double gb1 = 0., gb2 = 0., gw3 = 0., gb3 = 0., loss = 0.;
  for (int64_t base = (int64_t)blockIdx.x * 16; base < n; base += (int64_t)gridDim.x * 16) {
    if (xs_s < 16) xs[xs_s][xs_k] = base + xs_s < n ? eff(((double)nx - mu) / sd) : 0.;
    const float tgt[4] = {ny[0], ny[1], ny[2], ny[3]};
    fetch(base + (int64_t)gridDim.x * 16);
    __syncthreads();
    // forward
    double h1[4], h2[4], dz2[4], dz1[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      double z = b1;
#pragma unroll
      for (int k = 0; k < NIN; k++) z = fma(xs[4 * i + q][k], (double)w1[k], z);
      h1[i] = act64(z);
      h1q[4 * i + q][col] = (float)bf_hi((float)h1[i]);
    }
    __syncthreads();
    f64x4 z2 = {b2, b2, b2, b2};
#pragma unroll
    for (int st = 0; st < 16; st++)
      z2 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)h1q[r][4 * st + q], (double)w2[st], z2, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      h2[i] = act64(z2[i]);
      double p = h2[i] * w3;
#pragma unroll
      for (int off = 8; off >= 1; off >>= 1) p += __shfl_xor(p, off, 64);
      if (r == 0) ys[w][4 * i + q] = p;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int s = 4 * i + q;
      const double y = b3 + ((ys[0][s] + ys[1][s]) + (ys[2][s] + ys[3][s]));
      const double res = base + s < n ? y - (double)tgt[i] : 0.;
      const double dy = 2. * res * inv_n;
      loss += res * res * loss_scale;
      gb3 += dy;
      gw3 += dy * h2[i];
      dz2[i] = dy * w3 * (1. - h2[i] * h2[i]);
      gb2 += dz2[i];
      dz2s[s][col] = dz2[i];
    }
    __syncthreads();
    // dz1 of columns col
    f64x4 dh = {0., 0., 0., 0.};
#pragma unroll
    for (int st = 0; st < 16; st++)
      dh = __builtin_amdgcn_mfma_f64_16x16x4f64(dz2s[r][4 * st + q], (double)w2t[st], dh, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      dz1[i] = dh[i] * (1. - h1[i] * h1[i]);
      gb1 += dz1[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const double x = r < NIN ? xs[4 * i + q][r & 7] : 0.;
      gW1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, dz1[i], gW1, 0, 0, 0);
#pragma unroll
      for (int kt = 0; kt < 4; kt++)
        gW2[kt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)h1q[4 * i + q][16 * kt + r], dz2[i], gW2[kt], 0, 0, 0);
    }
    __syncthreads();
  }
  // out: C layout, row 4 i + q of a 16-row tile, column col
  double *g = part + (int64_t)blockIdx.x * PART;
#pragma unroll
  for (int kt = 0; kt < 4; kt++)
#pragma unroll
    for (int i = 0; i < 4; i++) g[OFF_W2 + (16 * kt + 4 * i + q) * NH + col] = gW2[kt][i];
#pragma unroll
  for (int i = 0; i < NIN / 4; i++) g[OFF_W1 + (4 * i + q) * NH + col] = gW1[i];
#pragma unroll
  for (int off = 16; off <= 32; off <<= 1) {
    gb1 += __shfl_xor(gb1, off, 64);
    gb2 += __shfl_xor(gb2, off, 64);
    gw3 += __shfl_xor(gw3, off, 64);
    gb3 += __shfl_xor(gb3, off, 64);
    loss += __shfl_xor(loss, off, 64);
  }
  if (q == 0) {
    g[OFF_B1 + col] = gb1;
    g[OFF_B2 + col] = gb2;
    g[OFF_W3 + col] = gw3;
    if (threadIdx.x == 0) {
      g[OFF_B3] = gb3;
      g[NTRAIN] = loss;
    }
  }
}

// the nb partial sums of weight e added in a fixed order, eight threads a weight
// (128 sums are then one round of loads);
// ADAM: the step and the weight's BF16 copies, else the gradient into grad[].
// The last number is the loss, added to *loss (first: in its place).
constexpr int UPDATE_WAYS = 8;
template <bool ADAM>
__global__ void __launch_bounds__(64 * UPDATE_WAYS) k_mlp_update(MlpDev m, const double *__restrict__ part, int nb,
                                                                 double lr, double b1t, double b2t, int first,
                                                                 double *__restrict__ m1, double *__restrict__ m2,
                                                                 float *__restrict__ grad,
                                                                 double *__restrict__ loss) {
  __shared__ double sum[UPDATE_WAYS][64];
  const int c = threadIdx.x & 63, w = threadIdx.x >> 6, e = blockIdx.x * 64 + c;
  double s = 0.;
  if (e <= NTRAIN) {
    for (int b = w; b < nb; b += 16 * UPDATE_WAYS) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; u++)
        v[u] = b + u * UPDATE_WAYS < nb ? part[(int64_t)(b + u * UPDATE_WAYS) * PART + e] : 0.;
#pragma unroll
      for (int u = 0; u < 16; u++) s += v[u];
    }
  }
  sum[w][c] = s;
  __syncthreads();
  if (w != 0 || e > NTRAIN) return;
  double gs = 0.;
#pragma unroll
  for (int u = 0; u < UPDATE_WAYS; u++) gs += sum[u][c];
  if (e == NTRAIN) {
    *loss = first ? gs : *loss + gs;
  } else if (ADAM) {
    const double b1 = 0.9, b2 = 0.999, eps = 1e-8;
    const double mm = b1 * m1[e] + (1. - b1) * gs, vv = b2 * m2[e] + (1. - b2) * gs * gs;
    m1[e] = mm;
    m2[e] = vv;
    // the weight is w + wlo, so that its steps do not round away
    const double wd = (double)m.w[e] + (double)m.wlo[e] - lr * (mm / (1. - b1t)) / (sqrt(vv / (1. - b2t)) + eps);
    const float v = (float)wd;
    m.w[e] = v;
    m.wlo[e] = (float)(wd - (double)v);
    refresh_bf16(e, v, m);
  } else {
    grad[e] = (float)gs;
  }
}

// the parameters a caller sets.  One that has the value it had keeps what its
// FP32 number rounds off, so that setting the parameters just read leaves a
// training as it is.
__global__ void k_mlp_set(MlpDev m, const float *__restrict__ src, float *__restrict__ zero) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= NPARAM) return;
  const float v = src[e];
  if (e < NTRAIN) {
    if (__float_as_int(v) != __float_as_int(m.w[e])) m.wlo[e] = 0.f;
    refresh_bf16(e, v, m);
    zero[e] = 0.f;
  }
  m.w[e] = v;
}

constexpr int COUNT_SLOTS = 64, COUNT_STRIDE = 8;

// ---------------------------------------------------------------------------
// inversion with the learned start.  The residual of the Newton system is
// evaluated in FP64 at the plain start (the reference's W from the previous
// primitives) and at the learned one, W_guess exp(y); the iteration starts
// from the smaller.  From there it is the mixed-precision inversion of
// HG_C2P_MIXED (FP32 Newton, FP64 and double-double polish, double-double
// primitives); a zone that does not converge joins the list that
// HG_C2P_REFINED inverts from the plain guess.  counts sums the zones solved from
// the learned start in COUNT_SLOTS parts a cache line apart: nearly every
// wavefront has some, and additions to one address are served one after
// another, 15 ns each, which was all that this kernel waited for: 2^20 zones 247 us
// in one part, 163 us in 64.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(64) k_c2p_learned(int64_t n, double gam, const double *__restrict__ U,
                                                    const double *__restrict__ gcov,
                                                    const double *__restrict__ gcon,
                                                    const double *__restrict__ gdet, double *__restrict__ pr,
                                                    int *__restrict__ pflag, int *__restrict__ iters, MlpDev m,
                                                    unsigned long long *__restrict__ ctr,
                                                    uint32_t *__restrict__ list,
                                                    unsigned long long *__restrict__ counts) {
  __shared__ float xin[64][NIN];
  __shared__ __align__(16) float h[16][NHS];
  __shared__ float yo[64];
  const int l = threadIdx.x;
  const int64_t t = (int64_t)blockIdx.x * 64 + l;
  const bool live = t < n;
  Geom G;
  double u[NPR], p[NPR], Ug[NPR];
  C2PInv c;
  double W_last = 1., alpha = 1.;
  int code = 1;
  if (live) {
    load_batch_zone(n, t, U, gcov, gcon, gdet, pr, G, u, p);
    code = c2p_setup_zone(u, G, gam, p, c, W_last, alpha, Ug);
    float x[NIN];
    c2p_features(c, W_last, alpha, gam, x);
#pragma unroll
    for (int k = 0; k < NIN; k++) xin[l][k] = (x[k] - m.w[OFF_MU + k]) / m.w[OFF_SD + k];
  } else {
#pragma unroll
    for (int k = 0; k < NIN; k++) xin[l][k] = 0.f;
  }
  __syncthreads();
  MlpRegs R;
  mlp_load(m, R);
  for (int g16 = 0; g16 < 4; g16++) {
    forward16(R, (const float(*)[NIN]) & xin[16 * g16][0], h, &yo[16 * g16]);
    __syncthreads();
  }
  const double igr = (gam - 1.0) / gam;
  bool fb = false, learned = false;
  if (live) {
#pragma unroll
    for (int i = B1; i <= B3; i++) p[i] = Ug[i];
    int it = 0, flag = code;
    if (code == 0) {
      double x0, x1;
      bool cand;
      it = learned_start(c, igr, W_last, yo[l], x0, x1, cand);
      fb = !mixed_zone(c, igr, x0, x1, p, it, flag);
      learned = cand && !fb;
    }
    if (!fb) {
      store_batch_zone(n, t, pr, p, code_assigns(flag));
      pflag[t] = flag;
      if (iters) iters[t] = it;
    }
  }
  list_append(fb, t, ctr, list);
  const unsigned long long ml = __ballot(learned);
  if (l == 0 && ml) atomicAdd(&counts[(blockIdx.x % COUNT_SLOTS) * COUNT_STRIDE], (unsigned long long)__popcll(ml));
}

}  // namespace

// one allocation holds everything: parameters, gradient, Adam moments, what the
// parameters round off and as many zeros (which stand for it in a gradient at
// the parameters themselves: a branch in the kernel costs a minibatch 1.2 us),
// the BF16 copies, the loss, the counts and the partial sums of the backward pass
struct hg_mlp {
  void *mem = nullptr;
  float *w = nullptr, *g = nullptr, *w2q = nullptr, *wlo = nullptr, *zero = nullptr;
  double *m1 = nullptr, *m2 = nullptr, *loss = nullptr, *part = nullptr;
  __bf16 *w1b = nullptr, *w2b = nullptr;
  unsigned long long *counts = nullptr;  // learned starts, in COUNT_SLOTS parts
  int step = 0;
};

static MlpDev dev_view(const hg_mlp *m) { return MlpDev{m->w, m->w1b, m->w2b, m->w2q, m->wlo}; }

// parameters from the host, through the room of the partial sums
static hipError_t upload_params(hg_mlp *m, const float *host) {
  hipError_t e = hipMemcpy(m->part, host, NPARAM * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_mlp_set, dim3((NPARAM + 255) / 256), dim3(256), 0, 0, dev_view(m), (const float *)m->part,
                     m->zero);
  e = hipGetLastError();
  return e == hipSuccess ? hipDeviceSynchronize() : e;
}

// blocks of the backward pass: one per 16-sample tile up to BACK_BLOCKS
static unsigned backward_blocks(int64_t n) {
  const int64_t tiles = (n + 15) / 16;
  return (unsigned)(tiles < BACK_BLOCKS ? tiles : BACK_BLOCKS);
}
constexpr unsigned UPDATE_BLOCKS = (NTRAIN + 1 + 63) / 64;

// the forward kernel's one-wavefront blocks: one per 16-sample tile up to
// 8192 (32 per CU), each then loops over its share of the tiles
static unsigned forward_blocks(int64_t n) {
  const int64_t tiles = (n + 15) / 16;
  return (unsigned)(tiles < 8192 ? tiles : 8192);
}

#define MLPCHECK(call)                                                              \
  do {                                                                              \
    hipError_t e_ = (call);                                                         \
    if (e_ != hipSuccess) {                                                         \
      set_error("%s:%d %s: %s", __FILE__, __LINE__, #call, hipGetErrorString(e_)); \
      return 1;                                                                     \
    }                                                                               \
  } while (0)

extern "C" int hg_mlp_destroy(hg_mlp *m) {
  if (!m) return 0;
  if (m->mem) (void)hipFree(m->mem);
  delete m;
  return 0;
}

extern "C" int hg_mlp_create(uint64_t seed, hg_mlp **out) {
  if (!out) { set_error("hg_mlp_create: null output"); return 1; }
  *out = nullptr;
  hg_mlp *m = new hg_mlp();
  std::vector<float> w(NPARAM, 0.f);
  // Glorot-uniform hidden weights from a 64-bit LCG; unit normalisation
  uint64_t s = seed * 6364136223846793005ull + 1442695040888963407ull;
  auto uni = [&]() {
    s = s * 6364136223846793005ull + 1442695040888963407ull;
    return (double)(s >> 11) * 0x1.0p-53;
  };
  double a1 = sqrt(6.0 / (NIN + NH)), a2 = sqrt(6.0 / (NH + NH)), a3 = sqrt(6.0 / (NH + 1));
  for (int e = 0; e < NIN * NH; e++) w[OFF_W1 + e] = (float)(a1 * (2 * uni() - 1));
  for (int e = 0; e < NH * NH; e++) w[OFF_W2 + e] = (float)(a2 * (2 * uni() - 1));
  for (int e = 0; e < NH; e++) w[OFF_W3 + e] = (float)(a3 * (2 * uni() - 1));
  for (int k = 0; k < NIN; k++) w[OFF_SD + k] = 1.f;
  // what starts as zero first
  const size_t np = (NPARAM + 63) / 64 * 64;
  size_t at = 0;
  auto take = [&at](size_t bytes) {
    const size_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  const size_t o_g = take(np * 4), o_m1 = take(np * 8), o_m2 = take(np * 8), o_wlo = take(np * 4),
               o_w1b = take(32 * NH * sizeof(__bf16)),
               o_w2b = take(NH * NH * sizeof(__bf16)), o_loss = take(sizeof(double)),
               o_counts = take(COUNT_SLOTS * COUNT_STRIDE * sizeof(unsigned long long)), zeroed = at, o_w = take(np * 4),
               o_w2q = take(NH * NH * sizeof(float)), o_part = take((size_t)BACK_BLOCKS * PART * sizeof(double)),
               o_zero = take(np * 4);
  hipError_t e = hipMalloc(&m->mem, at);
  if (e == hipSuccess) {
    char *b = (char *)m->mem;
    m->g = (float *)(b + o_g);
    m->m1 = (double *)(b + o_m1);
    m->m2 = (double *)(b + o_m2);
    m->wlo = (float *)(b + o_wlo);
    m->zero = (float *)(b + o_zero);
    m->w1b = (__bf16 *)(b + o_w1b);
    m->w2b = (__bf16 *)(b + o_w2b);
    m->loss = (double *)(b + o_loss);
    m->counts = (unsigned long long *)(b + o_counts);
    m->w = (float *)(b + o_w);
    m->w2q = (float *)(b + o_w2q);
    m->part = (double *)(b + o_part);
    e = hipMemset(m->mem, 0, zeroed);
  }
  if (e == hipSuccess) e = upload_params(m, w.data());
  if (e != hipSuccess) {
    set_error("hg_mlp_create: %s", hipGetErrorString(e));
    hg_mlp_destroy(m);
    return 1;
  }
  *out = m;
  return 0;
}

extern "C" int hg_mlp_nparams(void) { return NPARAM; }

extern "C" int hg_mlp_get_params(const hg_mlp *m, float *host) {
  if (!m || !host) { set_error("hg_mlp_get_params: null argument"); return 1; }
  MLPCHECK(hipMemcpy(host, m->w, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

extern "C" int hg_mlp_set_params(hg_mlp *m, const float *host) {
  if (!m || !host) { set_error("hg_mlp_set_params: null argument"); return 1; }
  for (int k = 0; k < NIN; k++)
    if (!(host[OFF_SD + k] > 0.f)) { set_error("hg_mlp_set_params: feature scales must be > 0"); return 1; }
  MLPCHECK(upload_params(m, host));
  return 0;
}

extern "C" int hg_mlp_features(int64_t n, double gam, const double *U, const double *gcov, const double *gcon,
                               const double *gdet, const double *p_guess, const double *p_solved, float *X,
                               float *y, int32_t *ok, void *stream) {
  if (n < 0 || (n > 0 && (!U || !gcov || !gcon || !gdet || !p_guess || !X || (y && !p_solved)))) {
    set_error("hg_mlp_features: bad arguments");
    return 1;
  }
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_mlp_features, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, gam, U, gcov, gcon,
                     gdet, p_guess, p_solved, X, y, ok);
  MLPCHECK(hipGetLastError());
  MLPCHECK(hipStreamSynchronize(s));
  return 0;
}

unsigned hg::group_blocks_mlp(const GridView &v) {
  return forward_blocks((int64_t)v.d.n1 * v.d.n2 * v.d.n3);
}

void hg::launch_group_mlp(const hg_mlp *m, const GridView *views, const unsigned *first, int n, unsigned total,
                          hipStream_t s) {
  if (total == 0) return;
  hipLaunchKernelGGL(kg_mlp_forward, dim3(total), dim3(64), 0, s, views, first, n, dev_view(m));
}

void hg::launch_mlp_forward(const hg_mlp *m, int64_t n, const float *X, float *y, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mlp_forward, dim3(forward_blocks(n)), dim3(64), 0, s, n, X, y, dev_view(m));
}

extern "C" int hg_mlp_forward(const hg_mlp *m, int64_t n, const float *X, float *y, void *stream) {
  if (!m || n < 0 || (n > 0 && (!X || !y))) { set_error("hg_mlp_forward: bad arguments"); return 1; }
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_mlp_forward, dim3(forward_blocks(n)), dim3(64), 0, s, n, X, y, dev_view(m));
  MLPCHECK(hipGetLastError());
  MLPCHECK(hipStreamSynchronize(s));
  return 0;
}

// gradients of the mean squared error over n samples (no update); grad_host
// (may be NULL) receives them, *loss the error
extern "C" int hg_mlp_gradient(hg_mlp *m, int64_t n, const float *X, const float *Y, float *grad_host,
                               float *loss, void *stream) {
  if (!m || n <= 0 || !X || !Y) { set_error("hg_mlp_gradient: bad arguments"); return 1; }
  hipStream_t s = (hipStream_t)stream;
  const unsigned nb = backward_blocks(n);
  MlpDev at = dev_view(m);
  at.wlo = m->zero;  // at the parameters that hg_mlp_get_params returns
  hipLaunchKernelGGL(k_mlp_backward, dim3(nb), dim3(256), 0, s, n, X, Y, at, 1.0 / (double)n,
                     1.0 / (double)n, m->part);
  hipLaunchKernelGGL(k_mlp_update<false>, dim3(UPDATE_BLOCKS), dim3(64 * UPDATE_WAYS), 0, s, at, (const double *)m->part,
                     (int)nb, 0., 0., 0., 1, m->m1, m->m2, m->g, m->loss);
  MLPCHECK(hipGetLastError());
  MLPCHECK(hipStreamSynchronize(s));
  if (grad_host) MLPCHECK(hipMemcpy(grad_host, m->g, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  double ls = 0.;
  if (loss) MLPCHECK(hipMemcpy(&ls, m->loss, sizeof ls, hipMemcpyDeviceToHost));
  if (loss) *loss = (float)ls;
  return 0;
}

// epochs of Adam over the n samples in minibatches of `batch` (in order);
// *loss receives the mean minibatch loss of the last epoch
extern "C" int hg_mlp_train_rate(hg_mlp *m, int64_t n, const float *X, const float *Y, int epochs, int batch,
                                 double rate, float *loss, void *stream) {
  if (!m || n <= 0 || !X || !Y || epochs < 0 || batch < 64) {
    set_error("hg_mlp_train: bad arguments (batch >= 64)");
    return 1;
  }
  hipStream_t s = (hipStream_t)stream;
  int64_t nb = (n + batch - 1) / batch;
  double last = 0.;
  for (int ep = 0; ep < epochs; ep++) {
    for (int64_t b = 0; b < nb; b++) {
      int64_t off = b * batch, cnt = (off + batch <= n) ? batch : n - off;
      const unsigned blocks = backward_blocks(cnt);
      hipLaunchKernelGGL(k_mlp_backward, dim3(blocks), dim3(256), 0, s, cnt, X + off * NIN, Y + off, dev_view(m),
                         1.0 / (double)cnt, 1.0 / (double)cnt / (double)nb, m->part);
      m->step++;
      const double b1t = pow(0.9, (double)m->step), b2t = pow(0.999, (double)m->step);
      hipLaunchKernelGGL(k_mlp_update<true>, dim3(UPDATE_BLOCKS), dim3(64 * UPDATE_WAYS), 0, s, dev_view(m),
                         (const double *)m->part, (int)blocks, rate, b1t, b2t, b == 0 ? 1 : 0, m->m1, m->m2, m->g,
                         m->loss);
    }
    MLPCHECK(hipGetLastError());
    MLPCHECK(hipMemcpyAsync(&last, m->loss, sizeof last, hipMemcpyDeviceToHost, s));
    MLPCHECK(hipStreamSynchronize(s));
  }
  if (loss) *loss = (float)last;
  return 0;
}

extern "C" int hg_mlp_train(hg_mlp *m, int64_t n, const float *X, const float *Y, int epochs, int batch, float lr,
                            float *loss, void *stream) {
  return hg_mlp_train_rate(m, n, X, Y, epochs, batch, (double)lr, loss, stream);
}

extern "C" int hg_utoprim_batch_learned(const hg_mlp *m, int64_t n, double gam, const double *U,
                                        const double *gcov, const double *gcon, const double *gdet,
                                        const double *gcovpert, double *pr, int32_t *pflag, int32_t *iters,
                                        int64_t *counts, void *stream) {
  (void)gcovpert;
  if (!m || n < 0 || n > (int64_t)0xFFFFFFFFll) { set_error("hg_utoprim_batch_learned: bad arguments"); return 1; }
  if (n == 0) {
    if (counts) counts[0] = counts[1] = 0;
    return 0;
  }
  if (!U || !gcov || !gcon || !gdet || !pr || !pflag) {
    set_error("hg_utoprim_batch_learned: null argument");
    return 1;
  }
  hipStream_t s = (hipStream_t)stream;
  // scratch of this call only (see hg_utoprim_batch)
  void *scr = nullptr;
  MLPCHECK(hipMallocAsync(&scr, c2p_scratch_bytes(n), s));
  unsigned long long *ctr = (unsigned long long *)scr;
  launch_c2p_reset(scr, s);
  hipError_t e = hipMemsetAsync(m->counts, 0, COUNT_SLOTS * COUNT_STRIDE * sizeof(unsigned long long), s);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_c2p_learned, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, n, gam, U, gcov, gcon, gdet,
                       pr, pflag, iters, dev_view(m), ctr, (uint32_t *)(ctr + C2P_NCTR), m->counts);
    if (launch_c2p_listed(n, gam, U, gcov, gcon, gdet, pr, pflag, iters, scr, s)) e = hipErrorUnknown;
  }
  unsigned long long h[COUNT_SLOTS * COUNT_STRIDE] = {}, len = 0;
  if (e == hipSuccess) e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(h, m->counts, sizeof h, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipMemcpyAsync(&len, ctr + C2P_LISTLEN, sizeof len, hipMemcpyDeviceToHost, s);
  hipError_t e2 = hipFreeAsync(scr, s);
  if (e == hipSuccess) e = e2;
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    set_error("hg_utoprim_batch_learned: %s", hipGetErrorString(e));
    return 1;
  }
  if (counts) {
    counts[0] = 0;
    for (int k = 0; k < COUNT_SLOTS; k++) counts[0] += (int64_t)h[k * COUNT_STRIDE];
    counts[1] = (int64_t)len;
  }
  return 0;
}
