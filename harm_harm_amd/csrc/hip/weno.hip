// weno.hip -- WENO5BND centre-to-edge reconstruction of the primitives as the
// reference compiles it for the torus (lim = WENO5BND): the whole storage line
// along a direction is reconstructed (slope_lim_linetype_c2e interpline.c:306)
// with
//   * the SMONO indicator (interpline.smono.c:198, :517): where the five-point
//     interpolant's first three derivatives at the neighbouring zone centres
//     agree in sign and are well above round-off, its face values replace
//     WENO's, with a linear ramp in between;
//   * WENO5 weights (compute_cf_stencil_weights reconstructeno.c:1693):
//     Jiang-Shu indicators of the point values, desensitised by eps |u|^2,
//     normalised, 1/(beta+eps)^2, normalised, limited (limit_weight :3015)
//     and normalised, with the SMONO ramp pulling them to equal (:852);
//   * the AND stencil reduction (compute_weights_ratios :2311): a zone whose
//     outer sub-stencils weigh 1.3-1.6 times more than the same three zones
//     weigh for the neighbours two zones away blends into WENO3;
//   * the pre/post-shock reduction (apply_additional_reduction_to_weights
//     :795): a zone whose pressure-jump measure dP exceeds 1/4 takes its
//     neighbours' reduction, fully at dP >= 1/2;
//   * the optimal face weights and the blend of WENO5, WENO3 and SMONO values
//     (choose_weno_order :2442, eno_cvt :884, eno_line_reconstruct :538).
//
// Device layout.  k_weno_dp forms dP for every direction at
// every zone that a face reconstruction needs (compute_df_line_new
// interpline.c:3557, from the zone's state and its two neighbours' along the
// direction).  Along x1, where a line is contiguous in memory,
// k_weno_recon_x1 gives each lane of a wave one zone of the line: the lane
// forms its zone's weights, takes its neighbours' from the lanes two away for
// the ratio test and the neighbours' ratios from the lanes one away, and
// writes the zone's faces (coalesced loads and stores, no carried state).
// Along x2 and x3, k_weno_recon sweeps segments of each storage line of one
// primitive in one thread (lanes are consecutive i: coalesced), carrying the
// last eight values and a four-zone pipeline of weights in registers.  The
// face-flux kernels read the left and right face values of zones -1 .. N
// back.  The arithmetic repeats the oracle's operation order (no contraction
// in this translation unit, correctly rounded quotients), so the face values
// agree bit for bit.
//
// The passes are bound by instruction issue: about 500 instructions a zone and
// primitive with 0.62 of the lanes active, 0.84 (x1), 0.75 and 0.63 (the sweeps
// alone on the chip) of the vector issue slots, an FP64 reciprocal taking four.
// Quotients are the largest part of it, so the weights of a zone share one
// reciprocal per normalisation (hd::recip, hd::quot), 7 + 3 + 3 instructions for
// three quotients instead of 33, and the SMONO and ratio tests settle clear
// cases without a quotient: on one state of the 256x128x64 torus the x1, x2 and x3
// passes took 265, 301 and 337 us so, 311, 405 and 450 with the compiler's
// divisions.  Alone on the chip they take 222, 227 and 175 us on the axisymmetric
// start and 298, 362 and 394 some twenty steps on, when most windows need weights.
#include <hip/hip_runtime.h>
#include <math.h>
#include <float.h>
#include <algorithm>
#include "dgrid.h"
#include "gkern.h"
#include "hhost.h"

namespace hk {
namespace {

using hd::Geom;
using hd::State;

constexpr double kSqrtWeps = 500.0 * DBL_EPSILON;  // SQRT_WENO_EPSILON
constexpr double kWeps = kSqrtWeps * kSqrtWeps;     // WENO_EPSILON = REDUCEEPSILON
constexpr double kMinNum = DBL_MIN;                 // MINNUMREPRESENT

constexpr double wmin(double a, double b) { return a < b ? a : b; }
constexpr double wmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double wminmod(double a, double b)
{
  return (a * b <= 0) ? 0.0 : ((fabs(a) < fabs(b)) ? a : b);
}

// get_sum_of_elements with SYMMETRIZE_WENO: mirror pairs first, the middle last
constexpr double sym3(double a0, double a1, double a2)
{
  double s = 0.0;
  s += a0 + a2;
  s += a1 * 1;
  return s;
}
constexpr double sym2(double a0, double a1)
{
  double s = 0.0;
  s += a0 + a1;
  s += a1 * 0;
  return s;
}
// the same sum of terms of which one at least is positive and none negative
// (the additions of 0 only matter for zeros' signs)
constexpr double sym3p(double a0, double a1, double a2) { return (a0 + a2) + a1; }
__device__ __forceinline__ double sym5(const double* a)
{
  double s = 0.0;
  s += a[0] + a[4];
  s += a[1] + a[3];
  s += a[2] * 1;
  return s;
}

template <int ORDER>
__device__ __forceinline__ double limit_weight(double w)
{
  const double avg = 1. / ORDER, w1 = 0.2 * avg, w2 = (1.0 - 0.2) * avg, w3 = (1.0 + 0.2) * avg, w4 = 1.0;
  if (w < w1) return 0.0;
  if (w < w2) return avg * (w - w1) / (w2 - w1);
  if (w < w3) return avg;
  return (w - w3) * (w4 - avg) / (w4 - w3) + avg;
}

// The same with one quotient by a constant: its numerator and denominator are
// picked by the branch w falls in (numerators are 0 or at least an ulp of w1,
// about 1e-17).
template <int ORDER>
__device__ __forceinline__ double limit_weight_q(double w)
{
  constexpr double avg = 1. / ORDER, w1 = 0.2 * avg, w2 = (1.0 - 0.2) * avg, w3 = (1.0 + 0.2) * avg, w4 = 1.0;
  constexpr double dlo = w2 - w1, dhi = w4 - w3, rlo = 1.0 / dlo, rhi = 1.0 / dhi;
  const bool hi = w >= w3;
  const double num = hi ? (w - w3) * (w4 - avg) : avg * (w - w1);
  const double q = hd::quot_const(num, hi ? dhi : dlo, hi ? rhi : rlo);
  double r = hi ? q + avg : w < w2 ? q : avg;
  return w < w1 ? 0.0 : r;
}

// Whether the unscaled quotients (dphys.h) of the indicators by their sum n can
// be used, with the factor sc for both.  Above 1e-200 the indicators are at
// least 1e-28 of n: each holds WENO_EPSILON (1.2e-26) times the window's sum of
// squares, and n is at most 60 times that sum.  Below (a field's front falls by
// some 1e-7 a zone, so most waves at it hold such a zone) the indicators and n,
// which is at least DBL_MIN, are brought up by a power of two, which leaves
// their quotients as they are (with the plain divisions there 30 steps of the
// 256x128x64 torus took 213.7 ms, so 206.1).  Beyond 1e200, infinities and NaN take the plain
// divisions.
__device__ __forceinline__ bool unscaled(double n, double& sc)
{
  sc = n < 1e-200 ? 0x1p600 : 1.0;
  return n < 1e200;
}

// The weights of the two uniform cases, formed by the same operations as the
// general code below (constant-folded, round to nearest):
//   * five equal values (below 1e100, where no square overflows): 3 u + u and
//     4 u round alike, or differ by an ulp whose square is 1e-5 of
//     WENO_EPSILON's part, so every weight is 1/3 to 1e-4 before limit_weight,
//     which maps all three to its flat band's value 1./3, and
//     (1/3 + 1/3) + 1/3 rounds to 1: the zone's weights are 1./3 each.  Its two
//     third-derivative estimates are each other's negatives, so its SMONO
//     indicator is 0.  (Axisymmetric regions along x3, and zero fields: with
//     the general code for all but zeros 30 steps of the 256x128x64 torus took
//     197.2 ms, so 194.5.)
//   * three equal values u[-1] = u[0] = u[1]: both WENO3 indicators are the
//     same, so both weights normalise to exactly 1/2, which limit_weight
//     keeps.
// The face weights of a zone whose unoptimized weights are 1./3 each, and
// the WENO3 face weights of 1/2 each, are these constants.
constexpr double kThird = 1. / 3;
constexpr double kL3n = sym3(kThird * (1. / 16.), kThird * (5. / 8.), kThird * (5. / 16.)) + kMinNum;
constexpr double kR3n = sym3(kThird * (5. / 16.), kThird * (5. / 8.), kThird * (1. / 16.)) + kMinNum;
constexpr double kL3[3] = {kThird * (1. / 16.) / kL3n, kThird * (5. / 8.) / kL3n, kThird * (5. / 16.) / kL3n};
constexpr double kR3[3] = {kThird * (5. / 16.) / kR3n, kThird * (5. / 8.) / kR3n, kThird * (1. / 16.) / kR3n};
constexpr double kL2n = sym2(0.5 * (1. / 4.), 0.5 * (3. / 4.)) + kMinNum;
constexpr double kR2n = sym2(0.5 * (3. / 4.), 0.5 * (1. / 4.)) + kMinNum;
constexpr double kL2[2] = {0.5 * (1. / 4.) / kL2n, 0.5 * (3. / 4.) / kL2n};
constexpr double kR2[2] = {0.5 * (3. / 4.) / kR2n, 0.5 * (1. / 4.) / kR2n};

// Unoptimized WENO5 weights of the zone u[0] (all three sub-stencils lie in
// the line for every zone the sweep computes).
__device__ __forceinline__ void weights3(const double* u, double* w)
{
  const double d10 = -(3 * u[0] + u[2]) + 4 * u[1], d11 = u[1] - u[-1], d12 = (3 * u[0] + u[-2]) - 4 * u[-1];
  const double d20 = (u[0] + u[2]) - 2 * u[1], d21 = (u[-1] + u[1]) - 2 * u[0], d22 = (u[0] + u[-2]) - 2 * u[-1];
  double s0 = 13. / 12. * d20 * d20 + 1. / 4. * d10 * d10;
  double s1 = 13. / 12. * d21 * d21 + 1. / 4. * d11 * d11;
  double s2 = 13. / 12. * d22 * d22 + 1. / 4. * d12 * d12;
  double q[5] = {u[-2] * u[-2], u[-1] * u[-1], u[0] * u[0], u[1] * u[1], u[2] * u[2]};
  const double err = sym5(q) * kWeps;
  s0 += err;
  s1 += err;
  s2 += err;
  double n = sym3(s0, s1, s2) + kMinNum, sc;
  if (unscaled(n, sc)) {
    // the quotients below stay between 1e-53 and 1e52 (t between WENO_EPSILON^2
    // = 1.5e-52 and about 1)
    const hd::Recip rn = hd::recip(n * sc);
    double t0 = hd::quot(s0 * sc, rn) + kWeps, t1 = hd::quot(s1 * sc, rn) + kWeps, t2 = hd::quot(s2 * sc, rn) + kWeps;
    t0 *= t0;
    t1 *= t1;
    t2 *= t2;
    const double w0 = hd::inv1(t0), w1 = hd::inv1(t1), w2 = hd::inv1(t2);
    const hd::Recip rw = hd::recip(sym3p(w0, w1, w2));
    const double l0 = limit_weight_q<3>(hd::quot(w0, rw)), l1 = limit_weight_q<3>(hd::quot(w1, rw)),
                 l2 = limit_weight_q<3>(hd::quot(w2, rw));
    const hd::Recip rl = hd::recip(sym3p(l0, l1, l2));  // the largest weight is at least 1/3, limited too
    w[0] = hd::quot(l0, rl);
    w[1] = hd::quot(l1, rl);
    w[2] = hd::quot(l2, rl);
    return;
  }
  s0 /= n;
  s1 /= n;
  s2 /= n;
  double t0 = s0 + kWeps, t1 = s1 + kWeps, t2 = s2 + kWeps;
  t0 *= t0;
  t1 *= t1;
  t2 *= t2;
  double w0 = 1. / t0, w1 = 1. / t1, w2 = 1. / t2;
  n = sym3(w0, w1, w2) + 0;
  w0 /= n;
  w1 /= n;
  w2 /= n;
  w0 = limit_weight<3>(w0);
  w1 = limit_weight<3>(w1);
  w2 = limit_weight<3>(w2);
  n = sym3(w0, w1, w2) + 0;
  w[0] = w0 / n;
  w[1] = w1 / n;
  w[2] = w2 / n;
}

// WENO3 weights, unoptimized then face-optimized ({1/4, 3/4} left, mirrored right)
__device__ __forceinline__ void weights2(const double* u, double* L2, double* R2)
{
  const double d0 = u[1] - u[0], d1 = u[0] - u[-1];
  double s0 = d0 * d0, s1 = d1 * d1;
  const double err = sym3(u[-1] * u[-1], u[0] * u[0], u[1] * u[1]) * kWeps;
  s0 += err;
  s1 += err;
  double n = sym2(s0, s1) + kMinNum, sc;
  if (unscaled(n, sc)) {  // as in weights3
    const hd::Recip rn = hd::recip(n * sc);
    double t0 = hd::quot(s0 * sc, rn) + kWeps, t1 = hd::quot(s1 * sc, rn) + kWeps;
    t0 *= t0;
    t1 *= t1;
    const double w0 = hd::inv1(t0), w1 = hd::inv1(t1);
    const hd::Recip rw = hd::recip(w0 + w1);
    const double m0 = limit_weight_q<2>(hd::quot(w0, rw)), m1 = limit_weight_q<2>(hd::quot(w1, rw));
    const hd::Recip rm = hd::recip(m0 + m1);
    const double v0 = hd::quot(m0, rm), v1 = hd::quot(m1, rm);
    const double l0 = v0 * (1. / 4.), l1 = v1 * (3. / 4.), r0 = v0 * (3. / 4.), r1 = v1 * (1. / 4.);
    const hd::Recip rl = hd::recip((l0 + l1) + kMinNum), rr = hd::recip((r0 + r1) + kMinNum);
    L2[0] = hd::quot(l0, rl);
    L2[1] = hd::quot(l1, rl);
    R2[0] = hd::quot(r0, rr);
    R2[1] = hd::quot(r1, rr);
    return;
  }
  s0 /= n;
  s1 /= n;
  double t0 = s0 + kWeps, t1 = s1 + kWeps;
  t0 *= t0;
  t1 *= t1;
  double w0 = 1. / t0, w1 = 1. / t1;
  n = sym2(w0, w1) + 0;
  w0 /= n;
  w1 /= n;
  w0 = limit_weight<2>(w0);
  w1 = limit_weight<2>(w1);
  n = sym2(w0, w1) + 0;
  w0 /= n;
  w1 /= n;
  double l0 = w0 * (1. / 4.), l1 = w1 * (3. / 4.), r0 = w0 * (3. / 4.), r1 = w1 * (1. / 4.);
  n = sym2(l0, l1) + kMinNum;
  L2[0] = l0 / n;
  L2[1] = l1 / n;
  n = sym2(r0, r1) + kMinNum;
  R2[0] = r0 / n;
  R2[1] = r1 / n;
}

// SMONO indicator (compute_mono_indicator_point_eno5).  The indicator is
// min over the three orders of |minmod(left, right)| against a round-off
// cut, clamped to [0, 1].  It is evaluated lazily, with the same values:
// minmod is 0 whenever its arguments are not strictly of one sign, and a
// quotient by 12 keeps its dividend's sign (or is 0), so an order whose
// numerators already disagree in sign gives 0 without its divisions; m = 0
// gives the indicator 0 and m >= cut gives 1 (m / cut >= 1 exactly).
__device__ __forceinline__ bool same_sign(double a, double b) { return (a > 0 && b > 0) || (a < 0 && b < 0); }
//
// Rounding is monotone, so the smallest of the quotients by 12 is the quotient
// of the smallest numerator: one division by 12 decides the indicator.  The
// minmods' sign products cannot underflow when the smallest estimate is above
// 1e-150; below that the estimates go through the minmods one by one.
__device__ __forceinline__ double smono_cut(const double* y, double m)
{
  const double norm = fabs(y[0]) + ((fabs(y[-1]) + fabs(y[1])) + (fabs(y[-2]) + fabs(y[2])));
  const double cut = norm * kSqrtWeps + kMinNum;
  if (m >= cut) return 1.0;
  return (m - 0.0) / (cut - 0.0);
}
__device__ __forceinline__ double smono(const double* y)
{
  const double L3 = (((-3 * y[-2] - y[2]) + (10 * y[-1] + 6 * y[1])) - 12 * y[0]) / 2.;
  const double R3 = (((y[-2] + 3 * y[2]) - (6 * y[-1] + 10 * y[1])) + 12 * y[0]) / 2.;
  if (!same_sign(L3, R3)) return 0.0;
  const double L2n = (((11 * y[-2] - y[2]) + (-20 * y[-1] + 4 * y[1])) + 6 * y[0]);
  const double R2n = (((-y[-2] + 11 * y[2]) + (4 * y[-1] - 20 * y[1])) + 6 * y[0]);
  if (!same_sign(L2n, R2n)) return 0.0;
  const double L1n = (((-3 * y[-2] + y[2]) + (-10 * y[-1] - 6 * y[1])) + 18 * y[0]);
  const double R1n = (((-y[-2] + 3 * y[2]) + (6 * y[-1] + 10 * y[1])) - 18 * y[0]);
  const double dl = y[-1] - y[-2], dr = y[2] - y[1];
  if (!same_sign(L1n, dl) || !same_sign(R1n, dr)) return 0.0;
  const double d3 = fmin(fabs(L3), fabs(R3)), d1 = fmin(fabs(dl), fabs(dr));
  const double n12 = fmin(fmin(fabs(L2n), fabs(R2n)), fmin(fabs(L1n), fabs(R1n)));
  const double m = fmin(fmin(hd::quot_const(n12, 12., 1. / 12.), d1), d3);
  if (m > 1e-150 && m < kBIG) {
    if (!same_sign(dl, dr)) return 0.0;
    return smono_cut(y, m);
  }
  const double m3 = fabs(wminmod(L3, R3));
  if (m3 == 0.0) return 0.0;
  const double L1 = wminmod(L1n / 12., dl);
  const double R1 = wminmod(R1n / 12., dr);
  const double m2 = fabs(wminmod(L2n / 12., R2n / 12.));
  double mm = kBIG;
  mm = wmin(mm, fabs(wminmod(L1, R1)));
  mm = wmin(mm, m2);
  mm = wmin(mm, m3);
  if (mm == 0.0) return 0.0;
  return smono_cut(y, mm);
}

// five-point interpolant at the left (RIGHT = false) or right face
template <bool RIGHT>
__device__ __forceinline__ double eno5(const double* y)
{
  double d[5];
  if (!RIGHT) {
    d[0] = -5. / 128. * y[-2];
    d[1] = 15. / 32. * y[-1];
    d[2] = 45. / 64. * y[0];
    d[3] = -5. / 32. * y[1];
    d[4] = 3. / 128. * y[2];
  } else {
    d[0] = 3. / 128. * y[-2];
    d[1] = -5. / 32. * y[-1];
    d[2] = 45. / 64. * y[0];
    d[3] = 15. / 32. * y[1];
    d[4] = -5. / 128. * y[2];
  }
  return sym5(d);
}

// eno_cvt of WENO5 (sub-stencil s covers u[-s .. 2-s]), zero-weight stencils skipped
template <bool RIGHT>
__device__ __forceinline__ double cvt3(const double* w, const double* u)
{
  double up0 = 0.0, up1 = 0.0, up2 = 0.0;
  if (!RIGHT) {
    if (w[0] != 0.0) up0 = w[0] * sym3(15. / 8. * u[0], -5. / 4. * u[1], 3. / 8. * u[2]);
    if (w[1] != 0.0) up1 = w[1] * sym3(3. / 8. * u[-1], 3. / 4. * u[0], -1. / 8. * u[1]);
    if (w[2] != 0.0) up2 = w[2] * sym3(-1. / 8. * u[-2], 3. / 4. * u[-1], 3. / 8. * u[0]);
  } else {
    if (w[0] != 0.0) up0 = w[0] * sym3(3. / 8. * u[0], 3. / 4. * u[1], -1. / 8. * u[2]);
    if (w[1] != 0.0) up1 = w[1] * sym3(-1. / 8. * u[-1], 3. / 4. * u[0], 3. / 8. * u[1]);
    if (w[2] != 0.0) up2 = w[2] * sym3(3. / 8. * u[-2], -5. / 4. * u[-1], 15. / 8. * u[0]);
  }
  return sym3(up0, up1, up2);
}
template <bool RIGHT>
__device__ __forceinline__ double cvt2(const double* w, const double* u)
{
  double up0 = 0.0, up1 = 0.0;
  if (!RIGHT) {
    if (w[0] != 0.0) up0 = w[0] * sym2(3. / 2. * u[0], -1. / 2. * u[1]);
    if (w[1] != 0.0) up1 = w[1] * sym2(1. / 2. * u[-1], 1. / 2. * u[0]);
  } else {
    if (w[0] != 0.0) up0 = w[0] * sym2(1. / 2. * u[0], 1. / 2. * u[1]);
    if (w[1] != 0.0) up1 = w[1] * sym2(-1. / 2. * u[-1], 3. / 2. * u[0]);
  }
  return sym2(up0, up1);
}

// What the sweep keeps of a zone between its weights and its face values:
// the unoptimized WENO5 weights after the SMONO ramp and the indicator.
// Everything else a zone's faces need (the SMONO face values, the WENO3
// weights, the optimized weights) is formed from the value window when its
// faces are, and the WENO3 weights only where the zone is reduced.
struct ZoneW {
  double u[3];
  double mono;
};

__device__ __forceinline__ void zone_weights(const double* y, ZoneW& z)
{
  if (y[-2] == y[0] && y[-1] == y[0] && y[1] == y[0] && y[2] == y[0] && fabs(y[0]) < 1e100) {
    z.mono = 0.0;
    z.u[0] = z.u[1] = z.u[2] = kThird;
    return;
  }
  z.mono = smono(y);
  if (z.mono == 1) {
    z.u[0] = z.u[1] = z.u[2] = 1.0 / 3;
  } else {
    weights3(y, z.u);
    if (z.mono > 0.0 && z.mono < 1.0)
#pragma unroll
      for (int s = 0; s < 3; s++) z.u[s] = (1.0 - z.mono) * z.u[s] + z.mono * (1.0 / 3);
  }
}

// one side of the AND ratio test: the zone's outer sub-stencil weight against
// the neighbour's weight of the same three zones (equal weights: exactly 1).
// Both lie in [WENO_EPSILON, 1 + WENO_EPSILON].
__device__ __forceinline__ double side_ratio(double uc, double un)
{
  if (uc == un) return 1.0;
  return hd::quot(uc + kWeps, hd::recip(un + kWeps));
}

// Lower-order fraction of a zone from its outer sub-stencil weights uc against
// the neighbours' un (a side that does not exist counts as BIG): the smaller
// ratio's place in the band 1.3 .. 1.6, clamped.  A ratio that is clearly at
// or below 1.3 on one side gives 0 without its quotient, two that are clearly
// at or above 1.6 give 1.
__device__ __forceinline__ double ratio_lof(double ucl, double unl, bool hasl, double ucr, double unr, bool hasr)
{
  const double min_rat = 1.3, max_rat = 1.6;
  if (!hasl && !hasr) return 1.0;
  const double al = ucl + kWeps, bl = unl + kWeps, ar = ucr + kWeps, br = unr + kWeps;
  if (hasr && ar <= 1.2999 * br) return 0.0;
  if (hasl && al <= 1.2999 * bl && !__builtin_isunordered(ar, br)) return 0.0;  // (a NaN on the right wins below)
  if ((!hasl || al >= 1.6001 * bl) && (!hasr || ar >= 1.6001 * br)) return 1.0;
  const double wl = hasl ? side_ratio(ucl, unl) : kBIG, wr = hasr ? side_ratio(ucr, unr) : kBIG;
  const double wrat = wmin(wl, wr);
  // the clamps below give exactly these at and beyond the band's ends
  if (wrat <= min_rat) return 0.0;
  if (wrat >= max_rat) return 1.0;
  double lof = (wrat - min_rat) / (max_rat - min_rat);
  lof = wmax(0., wmin(lof, 1.0));
  return wmax(lof, 0.0);  // the weights' own fraction starts at 0
}

// face values of zone y[0] from its kept weights, its final lower-order
// fraction and the SMONO ramp
__device__ __forceinline__ void zone_faces(const double* y, const ZoneW& z, double lof, double& lo, double& ro)
{
  const double m = z.mono;
  double ol = 0.0, orr = 0.0;
  if (m != 0) {
    ol = eno5<false>(y);
    orr = eno5<true>(y);
  }
  if (m >= 0.0 && m < 1.0) {
    // optimized WENO5 weights from the (ramped) unoptimized ones
    double L[3], R[3];
    if (z.u[0] == kThird && z.u[1] == kThird && z.u[2] == kThird) {
#pragma unroll
      for (int s = 0; s < 3; s++) {
        L[s] = kL3[s];
        R[s] = kR3[s];
      }
    } else {
      L[0] = z.u[0] * (1. / 16.);
      L[1] = z.u[1] * (5. / 8.);
      L[2] = z.u[2] * (5. / 16.);
      R[0] = z.u[0] * (5. / 16.);
      R[1] = z.u[1] * (5. / 8.);
      R[2] = z.u[2] * (1. / 16.);
      // the unoptimized weights are 0 or at least 1e-17 and sum to 1
      const hd::Recip rl = hd::recip(sym3p(L[0], L[1], L[2]) + kMinNum);
      const hd::Recip rr = hd::recip(sym3p(R[0], R[1], R[2]) + kMinNum);
#pragma unroll
      for (int s = 0; s < 3; s++) {
        L[s] = hd::quot(L[s], rl);
        R[s] = hd::quot(R[s], rr);
      }
    }
    double vl = 0.0, vr = 0.0;
    if (0.0 < lof) {
      double L2[2], R2[2];
      if (y[-1] == y[0] && y[0] == y[1]) {
        L2[0] = kL2[0];
        L2[1] = kL2[1];
        R2[0] = kR2[0];
        R2[1] = kR2[1];
      } else {
        weights2(y, L2, R2);
      }
#pragma unroll
      for (int s = 0; s < 3; s++) {
        L[s] *= (1. - lof);
        R[s] *= (1. - lof);
      }
#pragma unroll
      for (int s = 0; s < 2; s++) {
        L2[s] *= lof;
        R2[s] *= lof;
      }
      vl += cvt3<false>(L, y);
      vr += cvt3<true>(R, y);
      vl += cvt2<false>(L2, y);
      vr += cvt2<true>(R2, y);
    } else {
      vl += cvt3<false>(L, y);
      vr += cvt3<true>(R, y);
    }
    ol = (1.0 - m) * vl + m * ol;
    orr = (1.0 - m) * vr + m * orr;
  }
  lo = ol;
  ro = orr;
}

// dP terms of one zone along DIR (compute_df_line_new, b^dir b_t = 0)
struct DpTerms {
  double rho, par, veff, upar;
};
__device__ __forceinline__ DpTerms dp_terms(const State& q, const double* pr, const Geom& G, double gam, int dir)
{
  const double rho = pr[HARM_RHO], u = pr[HARM_UU];
  const double pgas = (gam - 1.0) * u;
  const double V = G.gdet * rho * q.ucon[dir];
  const double bsq = q.bsq, btt = 0.0;
  const double ptot = pgas + 0.5 * bsq;
  DpTerms t;
  t.rho = rho;
  t.par = fabs(q.p1ud0 * q.ucon[dir]);
  t.veff = copysign(1.0, V) * t.par / (sqrt(t.par) + D_SMALL);
  t.upar = fabs((u + pgas + bsq) * (fabs(q.ucon[dir]) * q.ucov[0]) + ptot + btt);
  return t;
}

__device__ __forceinline__ void load_prim(const double* __restrict__ p, long ncell, long c, double* pr)
{
#pragma unroll
  for (int v = 0; v < HARM_NPR; v++) pr[v] = p[v * ncell + c];
}

// dP of every active direction at the zones of z, -1 .. N of every active
// direction (the zones whose faces are reconstructed).  A zone's measure takes
// its own terms and those of its two neighbours along the direction.  A block
// marches through the k planes of a chunk with a tile of kDpI x kDpJ zones in
// (i, j), a halo zone on each active side included: every plane each thread
// forms the terms of its zone, the neighbours' of directions 1 and 2 come from
// LDS, the planes before and after from registers.
//
// Bound by the latency of a plane's chain at four waves a SIMD.  In two passes,
// the terms of every zone through memory (10 doubles written, 18 read), this
// took 94 + 54 us at 256x128x64, 23 + 16 at 128x64x64 and 8.4 + 5.2 at 97x51x22;
// so it takes 66, 26 and 11.4, though 40 % more terms are formed.  Tiles of
// 32 x 16 and 64 x 8: 76, 26, 11 and 86, 29, 11.  With the geometry read again
// every plane 108 us at four waves, 126 to 300 at six and eight (spills).
constexpr int kDpI = 32, kDpJ = 8;
struct DpPlan {
  int ti, tj, tk, nk;  // tiles along i, j; chunks along k, of nk planes
};
__global__ __launch_bounds__(kDpI* kDpJ) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_weno_dp(
    Dims d, Box z, DpPlan pl, const double* __restrict__ pb, const double* __restrict__ gcent, double gam,
    double* __restrict__ dp)
{
  __shared__ double lds[2][4][kDpI * kDpJ];  // by plane: veff, upar of direction 1, of direction 2
  const int e1 = d.n1 > 1, e2 = d.n2 > 1, e3 = d.n3 > 1;
  const int tid = threadIdx.x, ti = tid % kDpI, tj = tid / kDpI;
  int q = xcd_tile(blockIdx.x, gridDim.x);
  const int bi = q % pl.ti;
  q /= pl.ti;
  const int bk = q % pl.tk, bj = q / pl.tk;
  const int i = z.is - e1 + bi * (kDpI - 2 * e1) + ti, j = z.js - e2 + bj * (kDpJ - 2 * e2) + tj;
  const int k0 = z.ks + bk * pl.nk, k1 = min(k0 + pl.nk, z.ks + z.nk);  // planes k0 .. k1 - 1
  const bool act = i < z.is + z.ni + e1 && j < z.js + z.nj + e2;
  const bool out = act && ti >= e1 && ti < kDpI - e1 && tj >= e2 && tj < kDpJ - e2 && i < z.is + z.ni &&
                   j < z.js + z.nj;
  const long pp = act ? hd::pidx(d, i, j) : 0, nc = d.ncell;
  auto measure = [&](double rho, double par, double upar, double vp, double vm, double up, double um) {
    const double dv = vp - vm;
    return (fabs(rho * dv * dv) + fabs(up - um)) / (fabs(rho * par) + fabs(upar) + D_SMALL);
  };
  Geom G;
  hd::load_geom(gcent, pp, d.nplane, G);
  double rho1 = 0, par1 = 0, v1 = 0, u1 = 0, v2 = 0, u2 = 0;  // direction 3: the plane before, and the one before that
  double pr[HARM_NPR];
  long c = act ? hd::cidx(d, i, j, k0 - e3) : 0;
  load_prim(pb, nc, c, pr);
#pragma clang loop unroll(disable)
  for (int k = k0 - e3; k < k1 + e3; k++) {
    const int b = k & 1;
    DpTerms t[3];
    {
      State s;
      hd::get_state<false>(pr, G, gam, s);
#pragma unroll
      for (int dir = 1; dir <= 3; dir++) t[dir - 1] = dp_terms(s, pr, G, gam, dir);
    }
    const long cn = act ? c + (long)d.ps1 * d.ns2 : 0;
    if (k + 1 < k1 + e3) load_prim(pb, nc, cn, pr);
    lds[b][0][tid] = t[0].veff;
    lds[b][1][tid] = t[0].upar;
    lds[b][2][tid] = t[1].veff;
    lds[b][3][tid] = t[1].upar;
    __syncthreads();
    if (out && k >= k0 && k < k1) {
      if (e1)
        dp[c] = measure(t[0].rho, t[0].par, t[0].upar, lds[b][0][tid + 1], lds[b][0][tid - 1], lds[b][1][tid + 1],
                        lds[b][1][tid - 1]);
      if (e2)
        dp[nc + c] = measure(t[1].rho, t[1].par, t[1].upar, lds[b][2][tid + kDpI], lds[b][2][tid - kDpI],
                             lds[b][3][tid + kDpI], lds[b][3][tid - kDpI]);
    }
    if (e3 && out && k - 1 >= k0 && k - 1 < k1)
      dp[2 * nc + c - (long)d.ps1 * d.ns2] = measure(rho1, par1, u1, t[2].veff, v2, t[2].upar, u2);
    v2 = v1;
    u2 = u1;
    rho1 = t[2].rho;
    par1 = t[2].par;
    v1 = t[2].veff;
    u1 = t[2].upar;
    c = cn;
  }
}

// Segments of the storage lines along DIR (2 or 3), one primitive each, per
// thread.  Line index c = 0 .. n-1 is the sweep coordinate m = c - 4 (m = -4
// .. N+3); weights exist for c = 2 .. n-3, ratios for c = 2 .. n-3 (the left
// comparison from c = 4, the right one up to c = n-5), faces for c = 3 ..
// n-4 (m = -1 .. N).  A thread owns the faces of zones f0 .. f1 and starts
// five zones earlier so that the ratios of f0-1 and its neighbours exist.  At
// step s the value y[s] arrives, zone s-2 gets its weights, zone s-4 its
// ratio and zone s-5 its faces.  Threads are the lines of the face box's
// transverse plane with i fastest (no lanes padded per row); blockIdx.y is
// (primitive, segment).
template <int DIR>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_weno_recon(Dims d, Box b, int seg, const double* __restrict__ pb,
                                                         const double* __restrict__ dpd, double* __restrict__ L,
                                                         double* __restrict__ R)
{
  const int n0 = b.ni;
  const int n1 = DIR == 3 ? b.nj : b.nk;
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  if (t >= (long)n0 * n1) return;
  const int v = blockIdx.y % HARM_NPR, sg = blockIdx.y / HARM_NPR;
  const int t0 = (int)(t % n0), t1 = (int)(t / n0);
  int i, j, k;
  if (DIR == 2) { i = b.is + t0; j = -4; k = b.ks + t1; }
  else { i = b.is + t0; j = b.js + t1; k = -4; }
  const int N = DIR == 2 ? d.n2 : d.n3;
  const int n = N + 8;
  const int f0 = 3 + sg * seg, f1 = min(f0 + seg - 1, n - 4);
  const long st = DIR == 2 ? (long)d.ps1 : (long)d.ps1 * d.ns2;
  const long c0 = hd::cidx(d, i, j, k);
  const double* __restrict__ a = pb + (long)v * d.ncell + c0;
  double* __restrict__ Lo = L + (long)v * d.ncell + c0;
  double* __restrict__ Ro = R + (long)v * d.ncell + c0;
  const double* __restrict__ dpl = dpd + c0;

  double y[8];  // y[7] = y[s], y[0] = y[s-7]
#pragma unroll
  for (int m = 0; m < 8; m++) y[m] = 0.0;
  ZoneW zw[4] = {};  // zw[0] = zone s-2 ... zw[3] = zone s-5
  double z6u0 = 0.0;  // zone s-6's first weight (its ratio partner)
  double fd[3] = {0, 0, 0};  // ratio fractions of zones s-6, s-5, s-4
  const int s0 = max(0, f0 - 5);
  // the loads run two steps (values) and one step (dP) ahead of their use,
  // so that their latency overlaps a step's arithmetic
  double ya = s0 < n ? a[(long)s0 * st] : 0.0;
  double yb = s0 + 1 < n ? a[(long)(s0 + 1) * st] : 0.0;
  double dpa = s0 - 5 >= f0 ? dpl[(long)(s0 - 5) * st] : 0.0;
#pragma unroll 1
  for (int s = s0; s <= f1 + 5; s++) {
#pragma unroll
    for (int m = 0; m < 7; m++) y[m] = y[m + 1];
    y[7] = ya;
    ya = yb;
    yb = s + 2 < n ? a[(long)(s + 2) * st] : 0.0;
    const double dPi = dpa;
    dpa = (s + 1 - 5 >= f0 && s + 1 - 5 <= f1) ? dpl[(long)(s + 1 - 5) * st] : 0.0;
    // weights of zone s-2
    z6u0 = zw[3].u[0];
#pragma unroll
    for (int m = 3; m > 0; m--) zw[m] = zw[m - 1];
    if (s >= 4 && s <= n - 1 && s - 2 >= f0 - 3) zone_weights(y + 5, zw[0]);
    // ratio of zone r = s-4 (zw[2]) against zones r-2 (z6u0) and r+2 (zw[0])
    const int r = s - 4;
    fd[0] = fd[1];
    fd[1] = fd[2];
    fd[2] = 0.0;
    if (r >= 2 && r >= f0 - 1) {
      fd[2] = ratio_lof(zw[2].u[2], z6u0, r >= 4, zw[2].u[0], zw[0].u[2], r <= n - 5);
    }
    // faces of zone f = s-5 (zw[3], values y[0..4] centred on y[2])
    const int f = s - 5;
    if (f >= f0) {
      const double ss = wmin((fabs(dPi) - 0.5 * 0.5) / (0.5 * 0.5), 1.);
      double lof = fd[1];
      lof = wmax(lof, ss * fd[2]);
      lof = wmax(lof, ss * fd[0]);
      double lo, ro;
      zone_faces(y + 2, zw[3], lof, lo, ro);
      Lo[(long)f * st] = lo;
      Ro[(long)f * st] = ro;
    }
  }
}

// One zone per lane of a GL-lane group (g = 0 .. GL-1 its lane, c its line
// index, y[0..4] the values of zones c-2 .. c+2): the lane forms its zone's
// weights, then its ratio from the weights two lanes away, then its
// lower-order fraction from the ratios one lane away and its faces.  Lanes 3
// .. GL-4 of a group own faces (returns true and sets lo, ro); dp() reads the
// zone's dP and is called by those lanes only.  Every lane of the group must
// call it (the ratios travel by shuffles).  Same operations as the sweep.
template <int GL, class DP>
__device__ __forceinline__ bool lane_faces(const double* y, int c, int n, int g, bool act, DP dp, double& lo,
                                           double& ro)
{
  ZoneW z = {};
  if (act && c >= 2 && c <= n - 3) zone_weights(y + 2, z);
  // ratio of zone c against zones c-2 and c+2
  const double ul = __shfl_up(z.u[0], 2, GL), ur = __shfl_down(z.u[2], 2, GL);
  double fd = 0.0;
  if (act && c >= 2 && c <= n - 3 && g >= 2 && g <= GL - 3) {
    fd = ratio_lof(z.u[2], ul, c >= 4, z.u[0], ur, c <= n - 5);
  }
  const double fdm = __shfl_up(fd, 1, GL), fdp = __shfl_down(fd, 1, GL);
  if (act && c >= 3 && c <= n - 4 && g >= 3 && g <= GL - 4) {
    const double dPi = dp();
    const double ss = wmin((fabs(dPi) - 0.5 * 0.5) / (0.5 * 0.5), 1.);
    double lof = fd;
    lof = wmax(lof, ss * fdp);
    lof = wmax(lof, ss * fdm);
    zone_faces(y + 2, z, lof, lo, ro);
    return true;
  }
  return false;
}

// Direction 1 (lines contiguous in memory): a group of GL lanes holds GL
// consecutive zones c = (GL - 6) w + g of one storage line, so every load and
// store is contiguous; nw = ceil((n - 6) / (GL - 6)) groups cover a line.  A
// wave holds the same segment of two neighbouring lines j (same radii); the
// wave's segment, line pair, k and primitive are decoded once per wave in
// scalar registers.  (Along x2 and x3 the same scheme, with strided loads or
// staged through LDS, measured slower than the sweep.)
constexpr int kX1Lanes = 32;
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_weno_recon_x1(Dims d, Box b, int nw, const double* __restrict__ pb,
                                                            const double* __restrict__ dpd, double* __restrict__ L,
                                                            double* __restrict__ R)
{
  constexpr int GL = kX1Lanes;
  static_assert(64 / GL == 2, "two line groups per wave");
  const int njp = (b.nj + 1) / 2;
  const int wv = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)));
  if (wv >= njp * nw * b.nk * HARM_NPR) return;  // the whole wave is past the end
  int r = wv;
  const int jp = r % njp;
  r /= njp;
  const int ws = r % nw;
  r /= nw;
  const int kk = r % b.nk, v = r / b.nk;
  const int g = threadIdx.x & (GL - 1);
  const int jj = 2 * jp + ((threadIdx.x & 63) >= GL);
  const bool act = jj < b.nj;
  const int n = d.n1 + 8;
  const int c = (GL - 6) * ws + g;
  const long c0 = hd::cidx(d, -4, b.js + (act ? jj : b.nj - 1), b.ks + kk);
  const double* __restrict__ a = pb + (long)v * d.ncell + c0;

  double y[5];
#pragma unroll
  for (int m = 0; m < 5; m++) {
    const int cm = c - 2 + m;
    y[m] = (act && cm >= 0 && cm < n) ? a[cm] : 0.0;
  }
  double lo, ro;
  if (lane_faces<GL>(y, c, n, g, act, [&] { return dpd[c0 + c]; }, lo, ro)) {
    L[(long)v * d.ncell + c0 + c] = lo;
    R[(long)v * d.ncell + c0 + c] = ro;
  }
}

// Faces of storage lines along DIR for one primitive, a zone a thread.  Line
// index c = 0 .. n-1 is the coordinate m = c - 4 (m = -4 .. N+3); weights exist
// for c = 2 .. n-3, ratios for the same zones (the left comparison from c = 4,
// the right one up to c = n-5), faces for c = 3 .. n-4 (m = -1 .. N).  A block
// holds T consecutive zones, f0-3 .. f0+T-4, of several lines: each thread forms
// its zone's weights and leaves the two outer ones in LDS, then its ratio from
// the weights two zones away, then its faces from the ratios one zone away;
// the T - 6 inner zones own faces.  The lines are 8 consecutive i on 64-byte
// boundaries (the neighbouring block has the other half of each 128-byte row,
// on the same XCD).  LDS entries are numbered by thread, so a zone's
// neighbours along the line are a fixed distance away.
//
// For grids whose lines are too few to fill the chip with sweeps, which take a
// segment's zones one after the other: x2 + x3 take 59 + 62 us at 97x51x22 as
// sweeps and 31 + 29 so, 54 and 9 (x2) at 200x100x1, 68 + 68 and 53 + 45 at
// 96x64x32.  On large grids its barriers cost more than the sweeps' halo (waves
// in smooth regions wait for the others): 308 + 347 and 446 + 390 at 256x128x64,
// where smaller blocks change nothing (391 + 406 with 32 zones a segment).
// Whole RK3 steps of an evolved torus, where the directions share the chip, as
// sweeps and so: 96x64x32 981 and 953 us, 128x64x40 1349 and 1349, 200x40x50
// 1525 and 1507, 128x64x48 1523 and 1535, 128x64x64 1881 and 1968.
constexpr int kLineMax = 1024;  // threads of a block
constexpr int kCols = 8;        // lines of a block
struct LinePlan {
  int T, nseg;   // zones a segment (halo included), segments a line
  int nt, npl;   // line tiles, transverse planes
  int threads;
  long blocks;
};
template <int DIR>
__global__ __launch_bounds__(kLineMax) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_weno_line(
    Dims d, Box b, LinePlan pl, const double* __restrict__ pb, const double* __restrict__ dpd,
    double* __restrict__ L, double* __restrict__ R)
{
  constexpr int S = kCols;  // distance of neighbours along the line
  extern __shared__ double lds[];
  double *ru0 = lds, *ru2 = lds + blockDim.x, *rfd = lds + 2 * blockDim.x;
  const int tid = threadIdx.x;
  int q = xcd_tile(blockIdx.x, gridDim.x);
  const int tile = q % pl.nt;
  q /= pl.nt;
  const int sg = q % pl.nseg;
  q /= pl.nseg;
  const int plane = q % pl.npl, v = q / pl.npl;
  const int w = tid % kCols, l = tid / kCols;
  const int N = DIR == 2 ? d.n2 : d.n3, n = N + 8;
  const int c = sg * (pl.T - 6) + l;  // line index of this thread's zone
  const int i = -d.ng1 + tile * kCols + w;
  const int j = DIR == 2 ? -4 + c : b.js + plane, k = DIR == 2 ? b.ks + plane : -4 + c;
  const bool act = l < pl.T && c < n && i >= b.is && i < b.is + b.ni;
  const unsigned st = DIR == 2 ? (unsigned)d.ps1 : (unsigned)d.ps1 * d.ns2;
  const unsigned o = act ? (unsigned)hd::cidx(d, i, j, k) : 0u;  // (a plane stays below 2^29 elements)
  const double* __restrict__ a = pb + (long)v * d.ncell;
  const bool zone = act && c >= 2 && c <= n - 3;
  double y[5];
  ZoneW z = {};
  if (zone) {
#pragma unroll
    for (int m = 0; m < 5; m++) y[m] = a[o + (m - 2) * st];
    zone_weights(y + 2, z);
  }
  ru0[tid] = z.u[0];
  ru2[tid] = z.u[2];
  __syncthreads();
  double fd = 0.0;
  const bool ratio = zone && l >= 2 && l < pl.T - 2;
  if (ratio) {
    const bool hl = c >= 4, hr = c <= n - 5;
    fd = ratio_lof(z.u[2], ru0[hl ? tid - 2 * S : tid], hl, z.u[0], ru2[hr ? tid + 2 * S : tid], hr);
  }
  rfd[tid] = fd;
  __syncthreads();
  if (zone && l >= 3 && l < pl.T - 3 && c >= 3 && c <= n - 4) {
    const double dPi = dpd[o];
    const double ss = wmin((fabs(dPi) - 0.5 * 0.5) / (0.5 * 0.5), 1.);
    double lof = fd;
    lof = wmax(lof, ss * rfd[tid + S]);
    lof = wmax(lof, ss * rfd[tid - S]);
    double lo, ro;
    zone_faces(y + 2, z, lof, lo, ro);
    L[(long)v * d.ncell + o] = lo;
    R[(long)v * d.ncell + o] = ro;
  }
}

// Segments: as few as keep a block within its threads, of equal length, so the
// halo of six zones costs little (92 % of the threads own faces at 64 zones).
LinePlan plan_lines(int dir, const Dims& d, const Box& b)
{
  LinePlan p{};
  const int nf = (dir == 2 ? d.n2 : d.n3) + 2;  // faces of zones -1 .. N
  const int tmax = kLineMax / kCols;
  p.nseg = (nf + tmax - 7) / (tmax - 6);
  p.T = (nf + p.nseg - 1) / p.nseg + 6;
  p.npl = dir == 3 ? b.nj : b.nk;
  p.nt = (b.is + b.ni + d.ng1 + kCols - 1) / kCols;
  p.threads = (kCols * p.T + 63) / 64 * 64;
  p.blocks = (long)p.nt * p.nseg * p.npl * HARM_NPR;
  return p;
}

}  // namespace

// dP of every active direction over the zones the face reconstructions read
void launch_weno_dp(const Dims& d, hipStream_t s, const double* pb, const double* gcent, const Params& P, double* dp)
{
  const int e1 = d.n1 > 1, e2 = d.n2 > 1, e3 = d.n3 > 1;
  const Box z{-e1, -e2, -e3, d.n1 + 2 * e1, d.n2 + 2 * e2, d.n3 + 2 * e3};
  DpPlan pl;
  pl.ti = (z.ni + kDpI - 2 * e1 - 1) / (kDpI - 2 * e1);
  pl.tj = (z.nj + kDpJ - 2 * e2 - 1) / (kDpJ - 2 * e2);
  // chunks of at least two planes (a chunk forms the terms of two more), as
  // many as give the chip four blocks a CU
  const int want = (1024 + pl.ti * pl.tj - 1) / (pl.ti * pl.tj);
  pl.tk = std::max(1, std::min(want, z.nk / 2));
  pl.nk = (z.nk + pl.tk - 1) / pl.tk;
  pl.tk = (z.nk + pl.nk - 1) / pl.nk;
  hipLaunchKernelGGL(k_weno_dp, dim3((unsigned)(pl.ti * pl.tj * pl.tk)), dim3(kDpI * kDpJ), 0, s, d, z, pl, pb, gcent,
                     P.gam, dp);
}

// face values L, R (SoA like pb) of zones -1 .. N along dir over the
// transverse range of the face box b.
void launch_weno_recon(int dir, const Dims& d, const Box& b, hipStream_t s, const double* pb, const double* dp,
                       double* L, double* R)
{
  const double* dpd = dp + (long)(dir - 1) * d.ncell;
  if (dir == 1) {
    constexpr int GL = kX1Lanes;
    const int n = d.n1 + 8;
    const int nw = (n - 6 + GL - 7) / (GL - 6);
    const long nwave = (long)((b.nj + 1) / 2) * nw * b.nk * HARM_NPR;
    const long blocks = (nwave + kBlock / 64 - 1) / (kBlock / 64);
    hipLaunchKernelGGL(k_weno_recon_x1, dim3((unsigned)blocks), dim3(kBlock), 0, s, d, b, nw, pb, dpd, L, R);
    return;
  }
  // directions 2 and 3: lines cut into segments of at least kMinSeg faces,
  // about kWaveTarget waves in all: few enough that the five zones a segment
  // forms ahead of its faces cost little, and the other directions' passes fill
  // its last waves' place.  Steps of an evolved 256x128x64 torus with 2048,
  // 4096, 6144, 8192 and 16384: 5802, 5858, 5815, 5828 and 5940 us; of
  // 128x128x64: 3535, 3257, 3261, 3297 and 3299.
  constexpr long kWaveTarget = 6144;
  constexpr int kMinSeg = 16;
  const int N = dir == 2 ? d.n2 : d.n3;
  const int nf = N + 2;  // zones -1 .. N
  const long nl = (long)b.ni * (dir == 3 ? b.nj : b.nk);
  // a zone a thread where that makes at most 50 waves a SIMD (about 400 000 zones)
  constexpr long kLineWaves = 51200;
  if (nl * N * HARM_NPR <= 64 * kLineWaves) {
    const LinePlan p = plan_lines(dir, d, b);
    const dim3 grid((unsigned)p.blocks), blk((unsigned)p.threads);
    const size_t lds = sizeof(double) * 3 * p.threads;
    if (dir == 2) hipLaunchKernelGGL(k_weno_line<2>, grid, blk, lds, s, d, b, p, pb, dpd, L, R);
    if (dir == 3) hipLaunchKernelGGL(k_weno_line<3>, grid, blk, lds, s, d, b, p, pb, dpd, L, R);
    return;
  }
  const long waves1 = (nl * HARM_NPR + 63) / 64;
  int nseg = (int)std::max(1L, std::min((long)(nf / kMinSeg), (kWaveTarget + waves1 - 1) / waves1));
  const int seg = (nf + nseg - 1) / nseg;
  nseg = (nf + seg - 1) / seg;
  const dim3 grid((unsigned)((nl + kBlock - 1) / kBlock), (unsigned)(HARM_NPR * nseg));
  if (dir == 2) hipLaunchKernelGGL(k_weno_recon<2>, grid, dim3(kBlock), 0, s, d, b, seg, pb, dpd, L, R);
  if (dir == 3) hipLaunchKernelGGL(k_weno_recon<3>, grid, dim3(kBlock), 0, s, d, b, seg, pb, dpd, L, R);
}

}  // namespace hk
