// mlp.hip -- training and inference kernels of the learned inversion guess,
// and the batched inversion seeded by it.
//
// Training runs in one persistent workgroup (8 wavefronts) that loops over
// minibatches of 128 pairs: forward (three BF16 matrix products with FP32
// accumulation, tanh hidden layers), mean-squared error on the standardised
// targets, backward (the weight gradients as transposed products X^T G, the
// input gradients as G W^T), and Adam on an FP32 master copy.  Every gradient
// element is produced by exactly one lane with a fixed summation order, so a
// training run is bit-reproducible.
//
// The seeded inversion evaluates the network per wavefront on 64 zones (the
// matrix instructions need the whole wave, so every lane joins in, active or
// not), starts the FP64 Newton solve from the predicted W', and falls back to
// the plain guess for any zone whose seeded solve does not succeed.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>
#include <vector>
#include <algorithm>
#include "mlp.h"
#include "hhost.h"
#include "gkern.h"
#include "dinvert.h"

using hm::v4f;

struct harm_mlp {
  float* w32 = nullptr;     // kNParam master parameters
  float* adam_m = nullptr;  // first moments
  float* adam_v = nullptr;  // second moments
  uint16_t* wbf = nullptr;  // kNBf BF16 weight images
  float* norm = nullptr;    // kNNorm standardisation constants
  float* loss = nullptr;    // per-launch mean loss (device scalar)
  int64_t t = 0;            // Adam steps taken
  std::vector<float> hnorm; // host copy of norm
};

namespace {

constexpr int kBlock = 256;
constexpr int kBatch = 128;     // training minibatch
constexpr int kWaves = kBlock / 64;
using hm::v4s;

// ---------------------------------------------------------------------------
// shared pieces
// ---------------------------------------------------------------------------

// BF16 images of the weights from the FP32 parameters (the rows' padding zero).
__global__ void k_mlp_pack(const float* __restrict__ w, uint16_t* __restrict__ wbf)
{
  for (int e = threadIdx.x + blockIdx.x * blockDim.x; e < hm::kNBf; e += blockDim.x * gridDim.x) {
    float v = 0.0f;
    if (e < hm::kBfW2) {
      const int h = e / hm::kIn, f = e % hm::kIn;
      v = w[hm::kOffW1 + f * hm::kHid + h];
    } else if (e < hm::kBfW3) {
      const int x = e - hm::kBfW2, o = x / hm::kStride, h = x % hm::kStride;
      if (h < hm::kHid) v = w[hm::kOffW2 + h * hm::kHid + o];
    } else {
      const int x = e - hm::kBfW3, o = x / hm::kStride, h = x % hm::kStride;
      if (h < hm::kHid) v = w[hm::kOffW3 + h * hm::kOut + o];
    }
    wbf[e] = hm::f2bf(v);
  }
}

// What a forward pass reads, in LDS: the weight images and the biases of the
// three layers.
constexpr int kNBias = 2 * hm::kHid + 4;
struct __align__(16) Net {
  uint16_t w[hm::kNBf];
  float b[kNBias];
};

__device__ void stage_net(const uint16_t* __restrict__ wbf, const float* __restrict__ w32, Net& N)
{
  const uint4* src = (const uint4*)wbf;
  uint4* dst = (uint4*)N.w;
  for (int e = threadIdx.x; e < hm::kNBf / 8; e += blockDim.x) dst[e] = src[e];
  for (int e = threadIdx.x; e < hm::kHid; e += blockDim.x) {
    N.b[e] = w32[hm::kOffB1 + e];
    N.b[hm::kHid + e] = w32[hm::kOffB2 + e];
  }
  if (threadIdx.x < 4) N.b[2 * hm::kHid + threadIdx.x] = threadIdx.x < hm::kOut ? w32[hm::kOffB3 + threadIdx.x] : 0.0f;
}

// The network over a wave's 64 samples, lane l's raw features in f (zeros for
// a lane without one): output o (or, NOUT 1, output 0 alone) of the lane's own
// sample, standardised, in y[o].  The features pass between lanes through the
// wave's xs; each 16 samples stay in registers from there on, so the block
// needs no barrier.
template <int NOUT>
__device__ __forceinline__ void wave_net(const float* f, bool act, const float* __restrict__ norm, const Net& N,
                                         uint16_t (*xs)[hm::kIn], float* y)
{
  const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
  v4f lo, hi;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    lo[k] = act ? (f[k] - norm[k]) * norm[hm::kIn + k] : 0.0f;
    hi[k] = act ? (f[4 + k] - norm[4 + k]) * norm[hm::kIn + 4 + k] : 0.0f;
  }
  *(v4s*)&xs[l][0] = hm::f2bf4(lo);
  *(v4s*)&xs[l][4] = hm::f2bf4(hi);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll 1
  for (int m = 0; m < 4; m++) {
    v4s x = hm::frag(&xs[m * 16 + r][4 * (q & 1)]), h1[4], h2[4];
    if (q > 1) x = (v4s){0, 0, 0, 0};
    hm::layer1(x, N.w + hm::kBfW1, N.b, h1);
    hm::layer<4>(h1, N.w + hm::kBfW2, hm::kStride, N.b + hm::kHid, h2);
    const v4f acc = hm::layer3(h2, N.w + hm::kBfW3);
#pragma unroll
    for (int o = 0; o < NOUT; o++) {
      const float v = __shfl(acc[o] + N.b[2 * hm::kHid + o], r);
      if (q == m) y[o] = v;
    }
  }
}

// ---------------------------------------------------------------------------
// training pairs
// ---------------------------------------------------------------------------

// Features and targets of n inversion problems from their conserved state U
// (UEVOLVE, SoA), geometry (SoA) and converged primitives p (SoA).  X[z][8]
// raw features, T[z][2] = (log(W'/D), log(u~^2)), ok[z] = 1 when usable.
__global__ __launch_bounds__(kBlock) void k_mlp_pairs(const double* __restrict__ U, const double* __restrict__ geom,
                                                      const double* __restrict__ p, long n, double gam,
                                                      double gammafail, float* __restrict__ X,
                                                      float* __restrict__ T, int32_t* __restrict__ ok)
{
  const long z = (long)blockIdx.x * kBlock + threadIdx.x;
  if (z >= n) return;
  hd::Geom g;
  hd::load_geom(geom, z, n, g);
  const double ig = (g.gdet >= 0.0 ? 1.0 : -1.0) / (fabs(g.gdet) + D_SMALL);
  double Ut[HARM_NPR], pz[HARM_NPR];
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) {
    Ut[pl] = g.alpha * (U[pl * n + z] * ig);
    pz[pl] = p[pl * n + z];
  }
  hd::Inv s;
  double Qtcon[4], Bcon[4];
  hd::inv_setup(Ut, g, gam, gammafail, s, Qtcon, Bcon);
  float f[hm::kIn];
  hm::features(s, f);
  double Wp, utsq;
  hm::wp_of_prim(pz, g, s.D, gam, Wp, utsq);
  bool good = s.D > 0.0 && Wp > 0.0 && utsq >= 0.0 && isfinite(Wp) && isfinite(utsq);
  for (int k = 0; k < hm::kIn; k++) {
    good = good && isfinite(f[k]);
    X[z * hm::kIn + k] = f[k];
  }
  T[z * 2 + 0] = (float)log(Wp / s.D + hm::kTinyWp);
  T[z * 2 + 1] = (float)log(utsq + hm::kTinyUt);
  ok[z] = good ? 1 : 0;
}

// ---------------------------------------------------------------------------
// training (one persistent workgroup)
// ---------------------------------------------------------------------------
struct TrainArgs {
  float* w32;
  float* am;
  float* av;
  uint16_t* wbf;
  const float* norm;
  const float* X;
  const float* T;
  const int32_t* idx;  // sample order
  long nidx;
  long nx;             // rows of X and T
  long first;          // position in idx of this launch's first sample
  int nsteps;
  long t0;             // Adam steps before this launch
  float lr, beta1, beta2, eps;
  float* grad_out;     // UPDATE false: one batch's gradients, nothing else changed
  float* loss_out;     // mean loss over the launch's steps
};

constexpr int kTrainBlock = 512;
constexpr int kRow = kBatch + 8;  // a row of a transposed layer: 68 words, rows 4 banks apart
constexpr int kChunk = 16;        // steps whose loss sums and bias corrections are formed together

struct __align__(16) TrainLds {
  Net N;
  uint16_t w2[hm::kHid * hm::kStride];   // W2 [in][out], for the input gradients
  uint16_t w3[hm::kHid * hm::kOut];      // W3 [in][out]
  uint16_t x[2][kBatch * hm::kIn];       // this batch and the next: [sample][feature]
  uint16_t xT[2][hm::kIn * kRow];        // [feature][sample]
  uint16_t h1T[hm::kHid * kRow], h2T[hm::kHid * kRow];  // hidden layers, [unit][sample]
  uint16_t g1T[hm::kHid * kRow], g2T[hm::kHid * kRow];  // their gradients
  uint16_t dyT[hm::kOut * kRow];
  float dyf[hm::kOut][kBatch + 4];
  float t[2][kBatch * hm::kOut];
  float err[kChunk][kBatch * hm::kOut + 1];
  double bc[2 * kChunk][2];              // 1/(1 - beta^t) of two chunks
};

// sum of a row of 128 BF16 values in order
__device__ __forceinline__ float row_sum(const uint16_t* row)
{
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < kBatch / 8; c++) {
    const uint4 v = ((const uint4*)row)[c];
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      s += __uint_as_float(u[i] << 16);
      s += __uint_as_float(u[i] & 0xffff0000u);
    }
  }
  return s;
}

// A step is two phases with one barrier after each.  First each wave carries
// its 16 samples forward and back through the network in registers (hm::layer)
// and leaves the layers and their gradients transposed, sample fastest, in LDS;
// then 24 products over the 128 samples (16 of dW2, 4 of dW1, 4 of dW3), three
// a wave, the bias sums on one wave each, and Adam: parameters and moments stay
// in their lane's registers for the whole launch, LDS gets the BF16 images.
// The next batch's rows are fetched during the first phase and put into LDS in
// the second.  One compute unit works, so a step is bound by its issue slots
// (the hidden layers' 256 tanhs and Adam's 100 updates a wave) and by the
// latency of the chain through the two phases.
// 2000 steps over 2^18 pairs: 46 us a step with a 4-wave block that kept
// every layer in LDS at a stride of 64 (rows on one bank, two bytes a load) and
// the parameters in memory, 8.4 now.
template <bool UPDATE>
__global__ __launch_bounds__(kTrainBlock) void k_mlp_train(TrainArgs a)
{
  __shared__ TrainLds S;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, r = l & 15, q = l >> 4;
  stage_net(a.wbf, a.w32, S.N);

  // ---- the parameters this lane owns ----
  // W2 tiles 2w, 2w + 1: (in, out) = (16 (w/2) + 4 q + i, 16 (2 w % 4 + u) + r);
  // waves 0-3 W3: (in, out) = (16 w + 4 q + i, r), r < 2;
  // waves 4-7 W1: (feature, unit) = (4 q + i, 16 (w - 4) + r), q < 2;
  // waves 1, 2, 3: the biases of layers 1, 2, 3, one a lane
  const int in2 = 16 * (w >> 1) + 4 * q, out2 = 16 * (2 * w & 3) + r;
  const bool own3 = w < 4 && r < hm::kOut, own1 = w >= 4 && q < 2;
  const int off = w < 4 ? hm::kOffW3 + (16 * w + 4 * q) * hm::kOut + r : hm::kOffW1 + 4 * q * hm::kHid + 16 * (w - 4) + r;
  const int inc = w < 4 ? hm::kOut : hm::kHid;
  const bool ownb = w == 1 || w == 2 || (w == 3 && l < hm::kOut);
  const int offb = w == 1 ? hm::kOffB1 + l : w == 2 ? hm::kOffB2 + l : hm::kOffB3 + l;
  float w2[2][4], m2[2][4], v2[2][4], wo[4], mo[4], vo[4], wb = 0.f, mb = 0.f, vb = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int e = hm::kOffW2 + (in2 + i) * hm::kHid + out2 + 16 * u;
      w2[u][i] = a.w32[e];
      m2[u][i] = a.am[e];
      v2[u][i] = a.av[e];
      S.w2[(in2 + i) * hm::kStride + out2 + 16 * u] = hm::f2bf(w2[u][i]);
    }
    wo[i] = mo[i] = vo[i] = 0.f;
    if (own3 || own1) {
      wo[i] = a.w32[off + i * inc];
      mo[i] = a.am[off + i * inc];
      vo[i] = a.av[off + i * inc];
    }
    if (own3) S.w3[(16 * w + 4 * q + i) * hm::kOut + r] = hm::f2bf(wo[i]);
  }
  if (ownb) {
    wb = a.w32[offb];
    mb = a.am[offb];
    vb = a.av[offb];
  }

  // ---- the batch: sample tid - 384 in waves 6 and 7, a step ahead ----
  const int bs = tid - (kTrainBlock - kBatch);
  float fx[hm::kIn], ft[hm::kOut];
  long pos = 0, sidx = 0;
  const long hop = kBatch % a.nidx;
  auto next_index = [&]() {  // out-of-range indices are rejected on the host
    sidx = a.idx[pos];
    if (sidx < 0 || sidx >= a.nx) sidx = 0;
    pos += hop;
    if (pos >= a.nidx) pos -= a.nidx;
  };
  auto fetch = [&]() {
#pragma unroll
    for (int k = 0; k < hm::kIn; k++) fx[k] = a.X[sidx * hm::kIn + k];
#pragma unroll
    for (int o = 0; o < hm::kOut; o++) ft[o] = a.T[sidx * hm::kOut + o];
  };
  auto stage = [&](int b) {
    v4f lo, hi;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      lo[k] = (fx[k] - a.norm[k]) * a.norm[hm::kIn + k];
      hi[k] = (fx[4 + k] - a.norm[4 + k]) * a.norm[hm::kIn + 4 + k];
    }
    const v4s xl = hm::f2bf4(lo), xh = hm::f2bf4(hi);
    *(v4s*)&S.x[b][bs * hm::kIn] = xl;
    *(v4s*)&S.x[b][bs * hm::kIn + 4] = xh;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      S.xT[b][k * kRow + bs] = (uint16_t)xl[k];
      S.xT[b][(4 + k) * kRow + bs] = (uint16_t)xh[k];
    }
#pragma unroll
    for (int o = 0; o < hm::kOut; o++)
      S.t[b][bs * hm::kOut + o] = (ft[o] - a.norm[2 * hm::kIn + o]) / a.norm[2 * hm::kIn + hm::kOut + o];
  };
  auto corrections = [&](int step) {  // lane j: those of step + j
    if (l < kChunk) {
      const float t = (float)(a.t0 + step + l + 1);
      S.bc[(step + l) % (2 * kChunk)][0] = 1.0 / (1.0f - powf(a.beta1, t));
      S.bc[(step + l) % (2 * kChunk)][1] = 1.0 / (1.0f - powf(a.beta2, t));
    }
  };
  if (bs >= 0) {
    pos = (a.first + bs) % a.nidx;
    next_index();
    fetch();
    next_index();
    stage(0);
  }
  if (w == 0) corrections(0);
  float loss_acc = 0.0f;
  __syncthreads();

  for (int step = 0; step < a.nsteps; step++) {
    const int b = step & 1, slot = step % kChunk;
    if (bs >= 0) {
      fetch();
      next_index();
    }
    // ---- this wave's 16 samples, forward ----
    const int m = 16 * w + r;  // the lane's sample
    v4s x = hm::frag(&S.x[b][m * hm::kIn + 4 * (q & 1)]), h1[4], h2[4], g2[4];
    if (q > 1) x = (v4s){0, 0, 0, 0};
    auto put = [&](uint16_t* T, int t, v4s v) {
#pragma unroll
      for (int i = 0; i < 4; i++) T[(16 * t + 4 * q + i) * kRow + m] = (uint16_t)v[i];
    };
    hm::layer1(x, S.N.w + hm::kBfW1, S.N.b, h1);
    hm::layer<4>(h1, S.N.w + hm::kBfW2, hm::kStride, S.N.b + hm::kHid, h2);
    const v4f y = hm::layer3(h2, S.N.w + hm::kBfW3);
    // ---- the loss and its gradient: lanes q = 0, outputs in elements 0 and 1 ----
    v4f dyv = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int o = 0; o < hm::kOut; o++) {
      const float d = y[o] + S.N.b[2 * hm::kHid + o] - S.t[b][m * hm::kOut + o];
      dyv[o] = d * (2.0f / (kBatch * hm::kOut));
      if (q == 0) {
        S.err[slot][m * hm::kOut + o] = d * d;
        S.dyf[o][m] = dyv[o];
      }
    }
    v4s dy = hm::f2bf4(dyv);
    if (q > 0) dy = (v4s){0, 0, 0, 0};
    else {
      S.dyT[m] = (uint16_t)dy[0];
      S.dyT[kRow + m] = (uint16_t)dy[1];
    }
    // ---- back: dH2 = dY W3^T, dH1 = dZ2 W2^T ----
    auto through_tanh = [&](v4f g, v4s h) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float hf = hm::bf2f((uint16_t)h[i]);
        g[i] = g[i] * (1.0f - hf * hf);
      }
      return hm::f2bf4(g);
    };
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const uint32_t pair = *(const uint32_t*)&S.w3[(16 * t + r) * hm::kOut];
      v4s c = {(short)(pair & 0xffffu), (short)(pair >> 16), 0, 0};
      if (q > 0) c = (v4s){0, 0, 0, 0};
      v4f acc = {0.f, 0.f, 0.f, 0.f};
      acc = hm::mfma(c, dy, acc);
      g2[t] = through_tanh(acc, h2[t]);
      put(S.h1T, t, h1[t]);
      put(S.h2T, t, h2[t]);
      put(S.g2T, t, g2[t]);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
      v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; c++) acc = hm::mfma(hm::frag(&S.w2[(16 * t + r) * hm::kStride + 16 * c + 4 * q]), g2[c], acc);
      put(S.g1T, t, through_tanh(acc, h1[t]));
    }
    __syncthreads();
    // ---- gradients over the batch ----
    v4f d2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, dO = {0.f, 0.f, 0.f, 0.f};
    const uint16_t* ra = w < 4 ? &S.h2T[(16 * w + r) * kRow] : &S.xT[b][(r & 7) * kRow];
    const uint16_t* rb = w < 4 ? &S.dyT[(r & 1) * kRow] : &S.g1T[(16 * (w - 4) + r) * kRow];
#pragma unroll
    for (int c = 0; c < kBatch / 16; c++) {
      const int k = 16 * c + 4 * q;
      const v4s h = hm::frag(&S.h1T[(16 * (w >> 1) + r) * kRow + k]);
      d2[0] = hm::mfma(h, hm::frag(&S.g2T[out2 * kRow + k]), d2[0]);
      d2[1] = hm::mfma(h, hm::frag(&S.g2T[(out2 + 16) * kRow + k]), d2[1]);
      dO = hm::mfma(hm::frag(ra + k), hm::frag(rb + k), dO);
    }
    float gb = 0.0f;
    if (w == 1) gb = row_sum(&S.g1T[l * kRow]);
    else if (w == 2) gb = row_sum(&S.g2T[l * kRow]);
    else if (w == 3) {
      if (l < hm::kOut)
        for (int k = 0; k < kBatch; k++) gb += S.dyf[l][k];
    } else if (w == 0 && (slot == kChunk - 1 || step == a.nsteps - 1)) {
      float sl = 0.0f;
      if (l <= slot)
        for (int e = 0; e < kBatch * hm::kOut; e++) sl += S.err[l][e];
      for (int j = 0; j <= slot; j++) loss_acc += __shfl(sl, j) / (kBatch * hm::kOut);
      corrections(step + 1);
    }
    // ---- parameter step ----
    if constexpr (UPDATE) {
      const double rc1 = S.bc[step % (2 * kChunk)][0], rc2 = S.bc[step % (2 * kChunk)][1];
      // (float)(m rc) is m / (1 - beta^t) rounded once: a quotient of two 24-bit
      // numbers is never within 2^-49 of a tie, the product's error is 2^-52
      auto adam = [&](float& p, float& pm, float& pv, float g) {
        pm = a.beta1 * pm + (1.0f - a.beta1) * g;
        pv = a.beta2 * pv + (1.0f - a.beta2) * g * g;
        p = p - a.lr * (float)(pm * rc1) / (sqrtf((float)(pv * rc2)) + a.eps);
      };
#pragma unroll
      for (int u = 0; u < 2; u++) {
        v4f n;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          adam(w2[u][i], m2[u][i], v2[u][i], d2[u][i]);
          n[i] = w2[u][i];
        }
        const v4s nb = hm::f2bf4(n);
        *(v4s*)&S.N.w[hm::kBfW2 + (out2 + 16 * u) * hm::kStride + in2] = nb;
#pragma unroll
        for (int i = 0; i < 4; i++) S.w2[(in2 + i) * hm::kStride + out2 + 16 * u] = (uint16_t)nb[i];
      }
      if (own3 || own1) {
        v4f n;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          adam(wo[i], mo[i], vo[i], dO[i]);
          n[i] = wo[i];
        }
        const v4s nb = hm::f2bf4(n);
        if (own3) {
          *(v4s*)&S.N.w[hm::kBfW3 + r * hm::kStride + 16 * w + 4 * q] = nb;
#pragma unroll
          for (int i = 0; i < 4; i++) S.w3[(16 * w + 4 * q + i) * hm::kOut + r] = (uint16_t)nb[i];
        } else {
          *(v4s*)&S.N.w[hm::kBfW1 + (16 * (w - 4) + r) * hm::kIn + 4 * q] = nb;
        }
      }
      if (ownb) {
        adam(wb, mb, vb, gb);
        S.N.b[hm::kHid * (w - 1) + l] = wb;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int u = 0; u < 2; u++) a.grad_out[hm::kOffW2 + (in2 + i) * hm::kHid + out2 + 16 * u] = d2[u][i];
        if (own3 || own1) a.grad_out[off + i * inc] = dO[i];
      }
      if (ownb) a.grad_out[offb] = gb;
    }
    if (bs >= 0) stage(b ^ 1);
    __syncthreads();
  }
  if (tid == 0) a.loss_out[0] = loss_acc / a.nsteps;
  if constexpr (UPDATE) {
    // the parameters, their moments and the BF16 images back to memory
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int e = hm::kOffW2 + (in2 + i) * hm::kHid + out2 + 16 * u;
        a.w32[e] = w2[u][i];
        a.am[e] = m2[u][i];
        a.av[e] = v2[u][i];
      }
      if (own3 || own1) {
        a.w32[off + i * inc] = wo[i];
        a.am[off + i * inc] = mo[i];
        a.av[off + i * inc] = vo[i];
      }
    }
    if (ownb) {
      a.w32[offb] = wb;
      a.am[offb] = mb;
      a.av[offb] = vb;
    }
    for (int e = tid; e < hm::kNBf / 8; e += kTrainBlock) ((uint4*)a.wbf)[e] = ((const uint4*)S.N.w)[e];
  }
}

// ---------------------------------------------------------------------------
// inference
// ---------------------------------------------------------------------------
// X[n][8] raw features -> Y[n][2] raw predictions (log W'/D, log u~^2)
__global__ __launch_bounds__(kBlock) void k_mlp_forward(const uint16_t* __restrict__ wbf,
                                                        const float* __restrict__ w32, const float* __restrict__ norm,
                                                        const float* __restrict__ X, float* __restrict__ Y, long n)
{
  __shared__ Net N;
  __shared__ uint16_t xs[kWaves][64][hm::kIn];
  stage_net(wbf, w32, N);
  __syncthreads();
  const long z = (long)blockIdx.x * kBlock + threadIdx.x;
  float f[hm::kIn], y[hm::kOut];
#pragma unroll
  for (int k = 0; k < hm::kIn; k++) f[k] = z < n ? X[z * hm::kIn + k] : 0.0f;
  wave_net<hm::kOut>(f, z < n, norm, N, xs[threadIdx.x >> 6], y);
  if (z < n) {
#pragma unroll
    for (int o = 0; o < hm::kOut; o++)
      Y[z * 2 + o] = y[o] * norm[2 * hm::kIn + hm::kOut + o] + norm[2 * hm::kIn + o];
  }
}

// One zone's solve from W' = seed, or from the primitives' guess when plain:
// 0 done, 1 unfinished after `limit` iterations (ns unchanged), 2 the seeded
// solve failed (its strokes in ns) and the plain guess decides.
__device__ __forceinline__ int seeded_one(const double* __restrict__ U, const double* __restrict__ geom,
                                          double* __restrict__ p, int32_t* __restrict__ pflag,
                                          int32_t* __restrict__ niter, long n, double gam, double gammafail, long z,
                                          double seed, bool plain, int limit, int& ns)
{
  hd::Geom g;
  hd::load_geom(geom, z, n, g);
  double Uz[HARM_NPR], pz[HARM_NPR];
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) {
    Uz[pl] = U[pl * n + z];
    pz[pl] = p[pl * n + z];
  }
  const int ns0 = ns;
  bool solved;
  int fl = hd::utoprimgen<true>(Uz, g, gam, gammafail, pz, ns, plain ? __builtin_nan("") : seed, limit, &solved);
  if (fl == hd::kUnfinishedFlag) {
    ns = ns0;
    return 1;
  }
  if (!plain && fl != 0) return 2;
  if (!solved) {  // the guess stands (read again rather than kept through the iterations)
    const double* pr = hd::fresh(p);
#pragma unroll
    for (int pl = 0; pl <= HARM_U3; pl++) pz[pl] = pr[pl * n + z];
  }
  if (hd::needs_after_hot(fl, true, false)) {  // the cold retry, as harm_invert_batch
    double Ugf[HARM_NPR], p0[HARM_NPR];
    const double *pr = hd::fresh(p), *Ur = hd::fresh(U);
#pragma unroll
    for (int pl = 0; pl < HARM_NPR; pl++) {
      Ugf[pl] = Ur[pl * n + z];
      p0[pl] = pr[pl * n + z];
    }
    hd::load_geom(hd::fresh(geom), z, n, g);
    hd::geometry_free(Ugf, g, Ugf);
    fl = hd::after_hot(fl, Ugf, g, gam, gammafail, p0, pz, ns, true, false);
  }
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) p[pl * n + z] = pz[pl];
  pflag[z] = fl;
  if (niter) niter[z] = ns;
  return 0;
}

// Batched inversion started from the network's W' (harm_invert_batch's
// arguments, plus the count of zones that fell back to the plain guess), in
// rounds as k_invert_batch: a zone whose seeded solve is unfinished after
// kFirst iterations, or has failed, goes into the block's list with its seed
// and the strokes so far, and is solved in a full wave of such zones.
// 2^20 zones of a log-uniform sample take 0.84 ms (2.39 one zone a lane to the
// end, the plain solve in the same lane).
constexpr int kFirst = 16;
constexpr long kResident = 768;  // blocks the chip holds (three waves a SIMD)
constexpr int kPlain = 1 << 30;  // in a list entry: the seeded solve has failed
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_invert_batch_mlp(
    const uint16_t* __restrict__ wbf, const float* __restrict__ w32, const float* __restrict__ norm,
    const double* __restrict__ U, const double* __restrict__ geom, double* __restrict__ p,
    int32_t* __restrict__ pflag, int32_t* __restrict__ niter, long n, double gam, double gammafail, int rounds,
    unsigned long long* __restrict__ nfallback)
{
  __shared__ Net N;
  __shared__ uint16_t xs[kWaves][64][hm::kIn];
  __shared__ double lseed[2 * kBlock];
  __shared__ int list[2 * kBlock], lns[2 * kBlock];  // zones (from z0) to come back to, at most 255 + 256
  __shared__ int cnt;
  __shared__ unsigned int nfb;
  const int tid = threadIdx.x;
  const long z0 = (long)blockIdx.x * kBlock * rounds;
  const int first = rounds > 1 ? kFirst : 200;
  stage_net(wbf, w32, N);
  if (tid == 0) cnt = nfb = 0;
  __syncthreads();
  int round = 0;
#pragma clang loop unroll(disable)
  while (true) {
    const int c = __builtin_amdgcn_readfirstlane(cnt);  // the same in every thread: cnt changes between barriers only
    const bool more = round < rounds && z0 + (long)round * kBlock < n;
    if (!more && c == 0) break;
    const bool full = c >= kBlock || !more;
    int loc = -1, ns = 0;
    bool plain = false;
    double seed = 0.0;
    if (full) {
      if (tid < min(c, kBlock)) {
        const int e = c - 1 - tid;
        loc = list[e] & (kPlain - 1);
        plain = (list[e] & kPlain) != 0;
        seed = lseed[e];
        ns = lns[e];
      }
    } else {
      if (z0 + (long)round * kBlock + tid < n) loc = round * kBlock + tid;
      round++;
    }
    __syncthreads();  // the list's entries and cnt have been read
    if (full && tid == 0) cnt = c - min(c, kBlock);
    __syncthreads();
    if (!full) {  // the whole wave, for the matrix instructions
      float f[hm::kIn] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, y[1];
      double D = 1.0;
      if (loc >= 0) {
        const long z = z0 + loc;
        hd::Geom g;
        hd::load_geom(geom, z, n, g);
        const double ig = (g.gdet >= 0.0 ? 1.0 : -1.0) / (fabs(g.gdet) + D_SMALL);
        double Ut[HARM_NPR];
#pragma unroll
        for (int pl = 0; pl < HARM_NPR; pl++) Ut[pl] = g.alpha * (U[pl * n + z] * ig);
        hd::Inv s;
        double Qtcon[4], Bcon[4];
        hd::inv_setup(Ut, g, gam, gammafail, s, Qtcon, Bcon);
        hm::features(s, f);
        D = s.D;
      }
      wave_net<1>(f, loc >= 0, norm, N, xs[tid >> 6], y);
      const float y0 = y[0] * norm[2 * hm::kIn + hm::kOut] + norm[2 * hm::kIn];
      seed = D * exp((double)fminf(fmaxf(y0, -60.0f), 60.0f));
    }
    if (loc >= 0) {
      const int left = seeded_one(U, geom, p, pflag, niter, n, gam, gammafail, z0 + loc, seed, plain,
                                  full ? 200 : first, ns);
      if (left) {
        if (left == 2) atomicAdd(&nfb, 1u);
        const int e = atomicAdd(&cnt, 1);
        list[e] = loc | (left == 2 ? kPlain : 0);
        lseed[e] = seed;
        lns[e] = ns;
      }
    }
    __syncthreads();
  }
  if (nfallback && tid == 0 && nfb) atomicAdd(nfallback, (unsigned long long)nfb);
}

// deterministic host initialisation: Glorot-uniform weights, zero biases
void init_params(std::vector<float>& w, uint64_t seed)
{
  uint64_t s = seed * 0x9E3779B97F4A7C15ull + 0x1234567ull;
  auto uni = [&]() {
    s += 0x9E3779B97F4A7C15ull;
    uint64_t x = s;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    x ^= x >> 31;
    return (double)(x >> 11) * (1.0 / 9007199254740992.0);
  };
  w.assign(hm::kNParam, 0.0f);
  auto fill = [&](int off, int fin, int fout) {
    const double a = sqrt(6.0 / (fin + fout));
    for (int e = 0; e < fin * fout; e++) w[off + e] = (float)((2.0 * uni() - 1.0) * a);
  };
  fill(hm::kOffW1, hm::kIn, hm::kHid);
  fill(hm::kOffW2, hm::kHid, hm::kHid);
  fill(hm::kOffW3, hm::kHid, hm::kOut);
}

harm_status pack(harm_mlp* m, hipStream_t s)
{
  hipLaunchKernelGGL(k_mlp_pack, dim3(8), dim3(kBlock), 0, s, m->w32, m->wbf);
  return hh::check_launch("k_mlp_pack");
}

// The step's inversion with the learned guess (harm_set_inversion_guess):
// the zones of k_invert in the same order; per wave the features of 64 zones
// go through the network on the matrix cores, each zone's Newton solve then
// starts from the predicted W' (falling back to the previous primitives when
// it fails).  Bound by issue, the network's tanhs about as much as the Newton
// iterations; without the floors and with the fallback as a second pass of one
// loop the solve fits three waves a SIMD (145 registers, 229 before): 12 steps
// of 128x64x64 28.6 -> 28.1 ms.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_invert_grid_mlp(
    const uint16_t* __restrict__ wbf, const float* __restrict__ w32, const float* __restrict__ norm, hd::Dims d,
    hk::Params P, const double* __restrict__ U, const double* __restrict__ pg, double* __restrict__ pf,
    int32_t* __restrict__ pflag, const double* __restrict__ gcent, int finalstep, unsigned long long* __restrict__ di)
{
  __shared__ Net N;
  __shared__ uint16_t xs[kWaves][64][hm::kIn];
  stage_net(wbf, w32, N);
  __syncthreads();
  const int lb = hk::xcd_tile(blockIdx.x, gridDim.x);
  const int t = lb * kBlock + threadIdx.x;
  const bool act = t < d.n1 * d.n2 * d.n3;
  long o = 0, pp = 0;
  double D = 1.0;
  float y[1];
  {
    float f[hm::kIn] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (act) {
      int i, j, k;
      hk::zone_ijk(d, t, i, j, k);
      o = hd::cidx(d, i, j, k);
      pp = hd::pidx(d, i, j);
      hd::Geom g;
      hd::load_geom(gcent, pp, d.nplane, g);
      const double ig = (g.gdet >= 0.0 ? 1.0 : -1.0) / (fabs(g.gdet) + D_SMALL);
      double Ut[HARM_NPR];
#pragma unroll
      for (int pl = 0; pl < HARM_NPR; pl++) Ut[pl] = g.alpha * (U[pl * d.ncell + o] * ig);
      hd::Inv s;
      double Qtcon[4], Bcon[4];
      hd::inv_setup(Ut, g, P.gam, P.gammafail, s, Qtcon, Bcon);
      hm::features(s, f);
      D = s.D;
    }
    wave_net<1>(f, act, norm, N, xs[threadIdx.x >> 6], y);
  }
  int ns = 0, nf = 0, fb = 0;
  if (act) {
    const float y0 = y[0] * norm[2 * hm::kIn + hm::kOut] + norm[2 * hm::kIn];
    const double seed = D * exp((double)fminf(fmaxf(y0, -60.0f), 60.0f));
    const int fl = hk::invert_zone<true>(d, P, U, pg, pf, pflag, gcent, o, pp, ns, seed, &fb);
    nf = !finalstep && fl > 0;
  }
  hk::newton_counts_to(ns, nf, di, t, hk::fail_list_cap(d));
  __shared__ unsigned int nfb;
  if (threadIdx.x == 0) nfb = 0;
  __syncthreads();
  if (fb) atomicAdd(&nfb, 1u);
  __syncthreads();
  if (threadIdx.x == 0 && nfb) atomicAdd(&di[hk::DI_NFALLBACK], (unsigned long long)nfb);
}

}  // namespace

// ===========================================================================
// C ABI
// ===========================================================================
extern "C" harm_status harm_mlp_create(uint64_t seed, harm_mlp** out)
{
  if (!out) return hh::set_error(HARM_EINVAL, "harm_mlp_create: null argument");
  harm_mlp* m = new harm_mlp();
  auto fail = [&](harm_status st) {
    harm_mlp_destroy(m);
    return st;
  };
  harm_status st;
  if ((st = hh::check_hip(hipMalloc((void**)&m->w32, sizeof(float) * hm::kNParam), "hipMalloc")) != HARM_OK ||
      (st = hh::check_hip(hipMalloc((void**)&m->adam_m, sizeof(float) * hm::kNParam), "hipMalloc")) != HARM_OK ||
      (st = hh::check_hip(hipMalloc((void**)&m->adam_v, sizeof(float) * hm::kNParam), "hipMalloc")) != HARM_OK ||
      (st = hh::check_hip(hipMalloc((void**)&m->wbf, sizeof(uint16_t) * hm::kNBf), "hipMalloc")) != HARM_OK ||
      (st = hh::check_hip(hipMalloc((void**)&m->norm, sizeof(float) * hm::kNNorm), "hipMalloc")) != HARM_OK ||
      (st = hh::check_hip(hipMalloc((void**)&m->loss, sizeof(float) * 4), "hipMalloc")) != HARM_OK)
    return fail(st);
  std::vector<float> w;
  init_params(w, seed);
  std::vector<float> z(hm::kNParam, 0.0f);
  m->hnorm.assign(hm::kNNorm, 0.0f);
  for (int k = 0; k < hm::kIn; k++) m->hnorm[hm::kIn + k] = 1.0f;
  for (int o = 0; o < hm::kOut; o++) m->hnorm[2 * hm::kIn + hm::kOut + o] = 1.0f;
  if ((st = hh::check_hip(hipMemcpy(m->w32, w.data(), sizeof(float) * hm::kNParam, hipMemcpyHostToDevice), "init")) !=
          HARM_OK ||
      (st = hh::check_hip(hipMemcpy(m->adam_m, z.data(), sizeof(float) * hm::kNParam, hipMemcpyHostToDevice),
                          "init")) != HARM_OK ||
      (st = hh::check_hip(hipMemcpy(m->adam_v, z.data(), sizeof(float) * hm::kNParam, hipMemcpyHostToDevice),
                          "init")) != HARM_OK ||
      (st = hh::check_hip(hipMemcpy(m->norm, m->hnorm.data(), sizeof(float) * hm::kNNorm, hipMemcpyHostToDevice),
                          "init")) != HARM_OK ||
      (st = pack(m, nullptr)) != HARM_OK)
    return fail(st);
  if ((st = hh::check_hip(hipDeviceSynchronize(), "harm_mlp_create")) != HARM_OK) return fail(st);
  *out = m;
  return HARM_OK;
}

extern "C" harm_status harm_mlp_destroy(harm_mlp* m)
{
  if (!m) return HARM_OK;
  void* bufs[] = {m->w32, m->adam_m, m->adam_v, m->wbf, m->norm, m->loss};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  delete m;
  return HARM_OK;
}

extern "C" harm_status harm_mlp_get_params(harm_mlp* m, float* params, float* norm)
{
  if (!m) return hh::set_error(HARM_EINVAL, "harm_mlp_get_params: null handle");
  if (params) HH_HIP(hipMemcpy(params, m->w32, sizeof(float) * hm::kNParam, hipMemcpyDeviceToHost));
  if (norm) memcpy(norm, m->hnorm.data(), sizeof(float) * hm::kNNorm);
  return HARM_OK;
}

extern "C" harm_status harm_mlp_set_params(harm_mlp* m, const float* params, const float* norm)
{
  if (!m) return hh::set_error(HARM_EINVAL, "harm_mlp_set_params: null handle");
  if (params) {
    HH_HIP(hipMemcpy(m->w32, params, sizeof(float) * hm::kNParam, hipMemcpyHostToDevice));
    HH_TRY(pack(m, nullptr));
  }
  if (norm) {
    for (int k = 0; k < hm::kIn; k++)
      if (!(norm[hm::kIn + k] > 0.0f)) return hh::set_error(HARM_EINVAL, "harm_mlp_set_params: feature scale <= 0");
    for (int o = 0; o < hm::kOut; o++)
      if (!(norm[2 * hm::kIn + hm::kOut + o] > 0.0f))
        return hh::set_error(HARM_EINVAL, "harm_mlp_set_params: target spread <= 0");
    m->hnorm.assign(norm, norm + hm::kNNorm);
    HH_HIP(hipMemcpy(m->norm, norm, sizeof(float) * hm::kNNorm, hipMemcpyHostToDevice));
  }
  return hh::check_hip(hipDeviceSynchronize(), "harm_mlp_set_params");
}

extern "C" harm_status harm_mlp_pairs(const double* U, const double* geom, const double* p, int64_t n, double gam,
                                      double gammafail, float* X, float* T, int32_t* ok, void* stream)
{
  if (n <= 0 || !U || !geom || !p || !X || !T || !ok) return hh::set_error(HARM_EINVAL, "harm_mlp_pairs: bad arguments");
  const long nb = (long)((n + kBlock - 1) / kBlock);
  if (nb > 0x7fffffffL) return hh::set_error(HARM_EINVAL, "harm_mlp_pairs: n too large");
  hipLaunchKernelGGL(k_mlp_pairs, dim3((unsigned)nb), dim3(kBlock), 0, (hipStream_t)stream, U, geom, p, (long)n, gam,
                     gammafail, X, T, ok);
  return hh::check_launch("k_mlp_pairs");
}

extern "C" harm_status harm_mlp_fit_norm(harm_mlp* m, const float* X, const float* T, const int32_t* ok, int64_t n)
{
  if (!m || !X || !T || !ok || n <= 0) return hh::set_error(HARM_EINVAL, "harm_mlp_fit_norm: bad arguments");
  std::vector<float> hx((size_t)n * hm::kIn), ht((size_t)n * hm::kOut);
  std::vector<int32_t> hok(n);
  HH_HIP(hipMemcpy(hx.data(), X, hx.size() * sizeof(float), hipMemcpyDeviceToHost));
  HH_HIP(hipMemcpy(ht.data(), T, ht.size() * sizeof(float), hipMemcpyDeviceToHost));
  HH_HIP(hipMemcpy(hok.data(), ok, hok.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
  double s1[hm::kIn + hm::kOut] = {0}, s2[hm::kIn + hm::kOut] = {0};
  long cnt = 0;
  for (int64_t z = 0; z < n; z++) {
    if (!hok[z]) continue;
    cnt++;
    for (int k = 0; k < hm::kIn; k++) { s1[k] += hx[z * hm::kIn + k]; s2[k] += (double)hx[z * hm::kIn + k] * hx[z * hm::kIn + k]; }
    for (int o = 0; o < hm::kOut; o++) {
      s1[hm::kIn + o] += ht[z * 2 + o];
      s2[hm::kIn + o] += (double)ht[z * 2 + o] * ht[z * 2 + o];
    }
  }
  if (cnt < 2) return hh::set_error(HARM_EINVAL, "harm_mlp_fit_norm: fewer than two usable pairs");
  std::vector<float> nm(hm::kNNorm);
  for (int k = 0; k < hm::kIn + hm::kOut; k++) {
    const double mean = s1[k] / cnt, var = std::max(s2[k] / cnt - mean * mean, 1e-12);
    const double sd = sqrt(var);
    if (k < hm::kIn) { nm[k] = (float)mean; nm[hm::kIn + k] = (float)(1.0 / sd); }
    else { nm[2 * hm::kIn + (k - hm::kIn)] = (float)mean; nm[2 * hm::kIn + hm::kOut + (k - hm::kIn)] = (float)sd; }
  }
  return harm_mlp_set_params(m, nullptr, nm.data());
}

extern "C" harm_status harm_mlp_train(harm_mlp* m, const float* X, const float* T, int64_t nx, const int32_t* order,
                                      int64_t norder, int64_t first, int32_t nsteps, float lr, float* loss,
                                      void* stream)
{
  if (!m || !X || !T || nx <= 0 || !order || norder <= 0 || nsteps <= 0 || !(lr > 0.0f) || first < 0)
    return hh::set_error(HARM_EINVAL, "harm_mlp_train: bad arguments");
  TrainArgs a{};
  a.w32 = m->w32; a.am = m->adam_m; a.av = m->adam_v; a.wbf = m->wbf; a.norm = m->norm;
  a.X = X; a.T = T; a.nx = (long)nx; a.idx = order; a.nidx = (long)norder; a.first = (long)first; a.nsteps = nsteps;
  a.t0 = (long)m->t;
  a.lr = lr; a.beta1 = 0.9f; a.beta2 = 0.999f; a.eps = 1e-8f; a.grad_out = nullptr; a.loss_out = m->loss;
  hipLaunchKernelGGL(k_mlp_train<true>, dim3(1), dim3(kTrainBlock), 0, (hipStream_t)stream, a);
  HH_TRY(hh::check_launch("k_mlp_train"));
  m->t += nsteps;
  if (loss) {
    HH_HIP(hipStreamSynchronize((hipStream_t)stream));
    HH_HIP(hipMemcpy(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost));
  }
  return HARM_OK;
}

extern "C" harm_status harm_mlp_grad(harm_mlp* m, const float* X, const float* T, int64_t nx, const int32_t* order,
                                     float* grad, float* loss)
{
  if (!m || !X || !T || nx <= 0 || !order || !grad) return hh::set_error(HARM_EINVAL, "harm_mlp_grad: bad arguments");
  TrainArgs a{};
  a.w32 = m->w32; a.am = m->adam_m; a.av = m->adam_v; a.wbf = m->wbf; a.norm = m->norm;
  a.X = X; a.T = T; a.nx = (long)nx; a.idx = order; a.nidx = kBatch; a.first = 0; a.nsteps = 1; a.t0 = 0;
  a.lr = 0.0f; a.beta1 = 0.9f; a.beta2 = 0.999f; a.eps = 1e-8f; a.grad_out = grad; a.loss_out = m->loss;
  hipLaunchKernelGGL(k_mlp_train<false>, dim3(1), dim3(kTrainBlock), 0, nullptr, a);
  HH_TRY(hh::check_launch("k_mlp_train"));
  HH_HIP(hipDeviceSynchronize());
  if (loss) HH_HIP(hipMemcpy(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost));
  return HARM_OK;
}

extern "C" harm_status harm_mlp_forward(harm_mlp* m, const float* X, float* Y, int64_t n, void* stream)
{
  if (!m || !X || !Y || n <= 0) return hh::set_error(HARM_EINVAL, "harm_mlp_forward: bad arguments");
  const long nb = (long)((n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)nb), dim3(kBlock), 0, (hipStream_t)stream, m->wbf, m->w32, m->norm,
                     X, Y, (long)n);
  return hh::check_launch("k_mlp_forward");
}

extern "C" harm_status harm_invert_batch_mlp(harm_mlp* m, const double* U, const double* geom, double* p_inout,
                                             int32_t* pflag, int32_t* niter, int64_t n, double gam, double gammafail,
                                             unsigned long long* nfallback, void* stream)
{
  if (!m || n <= 0 || !U || !geom || !p_inout || !pflag)
    return hh::set_error(HARM_EINVAL, "harm_invert_batch_mlp: bad arguments");
  const long nb = (long)((n + kBlock - 1) / kBlock);
  if (nb > 0x7fffffffL) return hh::set_error(HARM_EINVAL, "harm_invert_batch_mlp: n too large");
  const int rounds = hh::inversion_rounds(nb, kResident);
  hipLaunchKernelGGL(k_invert_batch_mlp, dim3((unsigned)((nb + rounds - 1) / rounds)), dim3(kBlock), 0,
                     (hipStream_t)stream, m->wbf, m->w32, m->norm, U, geom, p_inout, pflag, niter, (long)n, gam,
                     gammafail, rounds, nfallback);
  return hh::check_launch("k_invert_batch_mlp");
}

harm_status hk::launch_invert_grid_mlp(const harm_mlp* m, const hd::Dims& d, const hk::Params& P, const double* U,
                                       const double* pg, double* pf, int32_t* pflag, const double* gcent,
                                       int finalstep, unsigned long long* di, hipStream_t s)
{
  const long nb = ((long)d.n1 * d.n2 * d.n3 + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_invert_grid_mlp, dim3((unsigned)nb), dim3(kBlock), 0, s, m->wbf, m->w32, m->norm, d, P, U, pg,
                     pf, pflag, gcent, finalstep, di);
  return hh::check_launch("k_invert_grid_mlp");
}
