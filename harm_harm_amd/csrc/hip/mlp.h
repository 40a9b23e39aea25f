// mlp.h -- the learned initial guess for the conserved-to-primitive inversion:
// an 8 -> 64 -> 64 -> 2 perceptron (tanh hidden layers) evaluated with BF16
// operands on the matrix cores (v_mfma_f32_16x16x16_bf16, FP32 accumulation).
//
// Inputs are eight scale-free functions of the invariants the 1-D W' Newton
// solve starts from (D, B^2, Q~^2, (Q.B)^2, Q.n; inv_setup in dphys.h); the
// two outputs are log(W'/D) and log(u~^2) of the solution, both standardised
// with the training set's mean and spread.  The Newton solve in FP64 stays the
// judge: the network only replaces the starting W'.
//
// The matrix instruction takes A(m, k) and B(k, n) as four consecutive k per
// lane and returns four consecutive rows of D per lane.  With the weights as A
// and the samples as B a layer's output tile is D(h, sample), which is the next
// layer's B as it stands: a wave carries 16 samples through the whole network
// in registers.  The weights are kept with k contiguous (transposed where that
// needs it), so every operand is one 8-byte load.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "dphys.h"

namespace hm {

constexpr int kIn = 8;     // input features
constexpr int kHid = 64;   // hidden width
constexpr int kOut = 2;    // outputs

// Parameter block (FP32 master copy), row-major [in][out]:
// W1[8][64] b1[64] W2[64][64] b2[64] W3[64][2] b3[2]
constexpr int kOffW1 = 0;
constexpr int kOffB1 = kOffW1 + kIn * kHid;
constexpr int kOffW2 = kOffB1 + kHid;
constexpr int kOffB2 = kOffW2 + kHid * kHid;
constexpr int kOffW3 = kOffB2 + kHid;
constexpr int kOffB3 = kOffW3 + kHid * kOut;
constexpr int kNParam = kOffB3 + kOut;  // 4866

// BF16 weight images, transposed so that the input runs fastest:
// W1T [64][8], W2T [64][72], W3T [2][72].  Rows of 72 values (36 words) put the
// 16 rows of an operand on different LDS banks.
constexpr int kStride = kHid + 8;
constexpr int kBfW1 = 0;
constexpr int kBfW2 = kBfW1 + kHid * kIn;
constexpr int kBfW3 = kBfW2 + kHid * kStride;
constexpr int kNBf = kBfW3 + kOut * kStride;  // 5264 bf16 values, whole 16-byte pieces

// standardisation: feature mean[8], feature scale[8] (1/std), target mean[2], target std[2]
constexpr int kNNorm = 2 * kIn + 2 * kOut;

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// float -> bf16, round to nearest even (NaN kept quiet)
__host__ __device__ inline uint16_t f2bf(float f)
{
  union { float f; uint32_t u; } v;
  v.f = f;
  if ((v.u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((v.u >> 16) | 0x40u);
  const uint32_t r = ((v.u >> 16) & 1u) + 0x7fffu;
  return (uint16_t)((v.u + r) >> 16);
}
__host__ __device__ inline float bf2f(uint16_t b)
{
  union { float f; uint32_t u; } v;
  v.u = (uint32_t)b << 16;
  return v.f;
}

// four consecutive k of an operand row, 8-byte aligned
__device__ __forceinline__ v4s frag(const uint16_t* p) { return *(const v4s*)p; }

// four floats to BF16, as f2bf but for the payload of a NaN
__device__ __forceinline__ v4s f2bf4(v4f f)
{
  typedef float v2f __attribute__((ext_vector_type(2)));
  typedef __bf16 v2b __attribute__((ext_vector_type(2)));
  union { v2b b[2]; v4s s; } u;
  u.b[0] = __builtin_convertvector((v2f){f[0], f[1]}, v2b);
  u.b[1] = __builtin_convertvector((v2f){f[2], f[3]}, v2b);
  return u.s;
}

// BF16 of tanhf of four values, the same bits as f2bf(tanhf(x)) in fewer
// instructions and without its branches.  Below 1/4 the series of tanh, above it 1 - 2/(exp(2x) + 1)
// with the hardware's exponential and reciprocal, each within 6 units of FP32's
// last place; a result that close to where BF16 rounding turns (24 of 65536)
// is computed again by tanhf.  Compared over all 2^32 arguments when it was
// written; a test keeps those around every rounding point of the range.  With it
// and the layers in registers the seeded inversion's 12 steps at 128 x 64 x 64
// take 30.9 ms, with tanhf and the layers in LDS 33.9.
__device__ __forceinline__ v4s tanh4(v4f x)
{
  constexpr unsigned kNear = 12;
  v4f t;
  bool near = false;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float a = fabsf(x[i]);
    const float e = __builtin_amdgcn_exp2f(a * 2.8853900817779268f);  // 2/ln 2
    const float big = fmaf(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f);
    const float y = a * a;
    float s = fmaf(y, 0.021869488f, -0.053968254f);  // 62/2835, -17/315
    s = fmaf(y, s, 0.13333333f);
    s = fmaf(y, s, -0.33333334f);
    const float small = fmaf(a * y, s, a);
    const float m = a < 0.25f ? small : big;
    near |= ((__float_as_uint(m) + 0x8000u + kNear) & 0xffffu) <= 2 * kNear;
    t[i] = copysignf(m, x[i]);
  }
  if (near) {
#pragma unroll 1
    for (int i = 0; i < 4; i++) {
      const float v = tanhf(i == 0 ? x[0] : i == 1 ? x[1] : i == 2 ? x[2] : x[3]);
      t[0] = i == 0 ? v : t[0];
      t[1] = i == 1 ? v : t[1];
      t[2] = i == 2 ? v : t[2];
      t[3] = i == 3 ? v : t[3];
    }
  }
  return f2bf4(t);
}

__device__ __forceinline__ v4f mfma(v4s a, v4s b, v4f acc)
{
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
}

// One wave's 16 samples through a layer of 64 outputs: lane l = 16 q + r holds
// of sample r the inputs 16 c + 4 q + i in in[c] and, on return, the outputs
// 16 c + 4 q + i in out[c].  W: the layer's image, rows of `stride`; b: biases.
template <int NC>
__device__ __forceinline__ void layer(const v4s* in, const uint16_t* W, int stride, const float* b, v4s* out)
{
  const int r = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int t = 0; t < kHid / 16; t++) {
    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; c++) acc = mfma(frag(W + (t * 16 + r) * stride + c * 16 + 4 * q), in[c], acc);
    const v4f bias = *(const v4f*)(b + t * 16 + 4 * q);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = acc[i] + bias[i];
    out[t] = tanh4(acc);
  }
}

// The first layer: 8 inputs of the 16 the instruction takes, the lanes of the
// other 8 (q > 1) holding zeros on both sides.  x: inputs 4 q + i of sample r.
__device__ __forceinline__ void layer1(v4s x, const uint16_t* W, const float* b, v4s* out)
{
  const int r = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int t = 0; t < kHid / 16; t++) {
    v4s w = frag(W + (t * 16 + r) * kIn + 4 * (q & 1));
    if (q > 1) w = (v4s){0, 0, 0, 0};
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    acc = mfma(w, x, acc);
    const v4f bias = *(const v4f*)(b + t * 16 + 4 * q);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = acc[i] + bias[i];
    out[t] = tanh4(acc);
  }
}

// The output layer, without its bias: in the lanes q = 0, output o of sample r
// in element o (the other rows of the product repeat the two weights' rows).
__device__ __forceinline__ v4f layer3(const v4s* in, const uint16_t* W)
{
  const int r = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
  v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < kHid / 16; c++) acc = mfma(frag(W + (r & 1) * kStride + c * 16 + 4 * q), in[c], acc);
  return acc;
}

__host__ __device__ inline double slog(double x) { return x >= 0.0 ? log1p(x) : -log1p(-x); }

// The eight raw features of an inversion problem (before standardisation).
// All are ratios to powers of D, so they do not depend on the density scale.
__device__ __forceinline__ void features(const hd::Inv& s, float* f)
{
  const double D = s.D > 0.0 ? s.D : D_SMALL;
  const double e = s.Qdotnp / D, q2 = s.Qtsq / (D * D), b2 = s.Bsq / D;
  const double qb2 = s.QdotBsq / (D * D * D);
  const double q = sqrt(fmax(q2, 0.0));
  double wcold = 0.0;  // the cold-hydro W'/D, a closed-form first estimate
  {
    const double det = 1.0 + q2;
    wcold = q2 / (1.0 + sqrt(det));
  }
  f[0] = (float)slog(e);
  f[1] = (float)slog(q2);
  f[2] = (float)slog(b2);
  f[3] = (float)slog(qb2);
  f[4] = (float)(q / (fabs(e) + 1.0 + q));
  f[5] = (float)(b2 / (b2 + fabs(e) + 1.0));
  f[6] = (float)(s.QdotBsq / (s.Qtsq * s.Bsq + D_SMALL));
  f[7] = (float)slog(wcold);
}

// W' of a primitive state in the frame of the solve (set_guess_Wp,
// utoprim_jon.c:1346): D u~^2/(1+gamma) + (u + p) gamma^2.
__device__ __forceinline__ void wp_of_prim(const double* prim, const hd::Geom& g, double D, double gam, double& Wp,
                                           double& utsq)
{
  utsq = 0.;
#pragma unroll
  for (int i = 1; i < 4; i++)
#pragma unroll
    for (int j = 1; j < 4; j++) utsq += hd::gco(g, i, j) * prim[HARM_U1 + i - 1] * prim[HARM_U1 + j - 1];
  const double gammasq = 1. + utsq;
  const double gamma = sqrt(gammasq);
  const double u = prim[HARM_UU];
  const double p = (gam - 1.0) * u;
  Wp = D * utsq / (1.0 + gamma) + (u + p) * gammasq;
}

// Floors of the target transforms (log of non-negative quantities).
constexpr double kTinyWp = 1e-14, kTinyUt = 1e-14;

}  // namespace hm
