// dinvert.h -- one zone of the step's inversion: Utoprimgen (utoprimgen.c:32:
// Jon's hot Newton solve, the inversion check and the cold retry as the
// configuration turns them on) and, on the final substep, fixup1zone's floors
// (fixup.c:561), as the inversion kernels of the step run it (the plain one in
// grid.hip, the learned-guess one in mlp.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "dgrid.h"
#include "gkern.h"

namespace hk {

using hd::Dims;
using hd::Geom;
using hd::State;

// dfl[pl] += dV (U(pa)[pl] - U(pb)[pl]), U with gdet: the conserved change of
// one fix as the energy file accounts it (diag_fixup, fixup.c:303-405)
__device__ __forceinline__ void fix_delta_to(const Params& P, const Geom& G, const double* pb, const double* pa,
                                             double* dfl)
{
  const double dV = P.dx[1] * P.dx[2] * P.dx[3];
  State q;
  double Ub[HARM_NPR], Ua[HARM_NPR];
  hd::get_state(pb, G, P.gam, q);
  hd::primtoflux(pb, q, 0, G, Ub);
  hd::get_state(pa, G, P.gam, q);
  hd::primtoflux(pa, q, 0, G, Ua);
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) dfl[pl] += dV * (Ua[pl] - Ub[pl]);
}

// ---------------------------------------------------------------------------
// inversion + fixup1zone (floors via ZAMO-frame mass/energy addition)
// ---------------------------------------------------------------------------
// fixup1zone on the final substep (fixup.c:561-830): the density and
// internal-energy floors (mass and energy added in the ZAMO frame, then the
// floors' own Utoprimgen from the primitives so far) and the Lorentz-factor
// limit, on the zone's primitives pf[pl * ncell + o], left in pz, with flag fl
// (replaced by the floors' inversion flag when the floors changed the zone).
// Returns the flag; the floors' Newton strokes are added to ns.  *changed
// reports whether pz differs from pf, which is not written.  The geometry and
// the primitives are read again after the solve (an L1/L2 hit) instead of
// holding 86 registers through the Newton iterations.
// DIAG (final substep): the states each fix started from are kept for the
// energy-file accounting (diag_fixup, fixup.c:220): fx_flag[o] gets bit 0
// when the floors changed the zone (fixup.c:766) and bit 1 when the gamma
// limit did (fixup.c:784); fx_p0 (SoA, stride ncell) then holds the
// primitives ahead of both fixes and, when the floors changed them, fx_pfl
// the primitives after the floors.  Only fixed zones store their states.
template <bool DIAG = false>
__device__ __forceinline__ int floors_zone(const Dims& d, const Params& P, const double* __restrict__ gcent,
                                           const double* __restrict__ floors, const double* pf,
                                           double* pz, int fl, long o, long pp, int& ns, bool* changed,
                                           double* __restrict__ fx_p0, double* __restrict__ fx_pfl,
                                           uint8_t* __restrict__ fx_flag)
{
  const long nc = d.ncell;
  Geom G;
  hd::load_geom(gcent, pp, d.nplane, G);
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) pz[pl] = pf[pl * nc + o];
  auto floor_of = [&](const double* __restrict__ fls, int pl) {
    const double v = fls[pl * d.nplane + pp];
    return v < D_SMALL ? D_SMALL : v;
  };
  bool didchange = false;
  double dpr[HARM_NPR];
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) {
    const double fv = pl <= HARM_UU ? floor_of(floors, pl) : 0.0;
    const bool below = pl <= HARM_UU && fv > pz[pl];
    didchange = didchange || below;
    dpr[pl] = below ? fv - pz[pl] : 0.0;
  }
  if (didchange) {
    if (DIAG) {
#pragma unroll
      for (int pl = 0; pl < HARM_NPR; pl++) fx_p0[pl * nc + o] = pz[pl];
    }
    Geom G1 = G;
    G1.gdet = 1.0;
    State q, dq;
    double Ua[HARM_NPR], dUa[HARM_NPR];
    hd::get_state(pz, G, P.gam, q);
    hd::primtoflux(pz, q, 0, G1, Ua);
    hd::get_state(dpr, G, P.gam, dq);
    hd::primtoflux(dpr, dq, 0, G1, dUa);
#pragma unroll
    for (int pl = 0; pl < HARM_NPR; pl++) Ua[pl] += dUa[pl];
    // the floors' own Utoprimgen (UNOTHING), from the primitives so far;
    // any flag > 0, the cold retry's mark included, restores the floored
    // primitives
    bool solved;
    fl = hd::jon(Ua, G, P.gam, P.gammafail, pz, ns, __builtin_nan(""), 200, &solved);
    const double* pfr = hd::fresh(pf);
    if (!solved) {
#pragma unroll
      for (int pl = 0; pl <= HARM_U3; pl++) pz[pl] = pfr[pl * nc + o];
    }
    hd::load_geom(hd::fresh(gcent), pp, d.nplane, G);
    if (hd::needs_after_hot(fl, P.hot2cold, P.checkinv)) {
      double p0[HARM_NPR];
#pragma unroll
      for (int pl = 0; pl < HARM_NPR; pl++) p0[pl] = pfr[pl * nc + o];
      fl = hd::after_hot(fl, Ua, G, P.gam, P.gammafail, p0, pz, ns, P.hot2cold, P.checkinv);
    }
    if (fl > 0) {
#pragma unroll
      for (int pl = 0; pl < HARM_NPR; pl++) {
        pz[pl] = pfr[pl * nc + o];
        if (pl <= HARM_UU) {
          const double fv = floor_of(hd::fresh(floors), pl);
          if (fv > pz[pl]) pz[pl] = fv;
        }
      }
    }
  }
  double pb4[HARM_NPR];  // DIAG: the primitives ahead of the gamma limit
  if (DIAG) {
#pragma unroll
    for (int pl = 0; pl < HARM_NPR; pl++) pb4[pl] = pz[pl];
  }
  const bool lg = hd::limit_gamma(P.gammamax, pz, G);
  if (DIAG) {
    if (lg) {
      double* dst = didchange ? fx_pfl : fx_p0;  // with no floor step these are also the primitives ahead of both
#pragma unroll
      for (int pl = 0; pl < HARM_NPR; pl++) dst[pl * nc + o] = pb4[pl];
    }
    fx_flag[o] = (uint8_t)((didchange ? 1 : 0) | (lg ? 2 : 0));
  }
  *changed = didchange || lg;
  return fl;
}

// One zone's solve: conserved U (with gdet) and the guess pg read at offset o,
// the result written to pf and pflag.  Returns the flag; the Newton stroke
// count is added to ns.  The floors and the Lorentz-factor limit of the final
// substep are a pass of their own (floors_zone), so that this solve keeps its
// registers.
//
// SEEDED: the Newton solve starts from W' = wp_seed (the learned guess); when
// that solve fails, the zone is solved again from the primitives' guess as
// the plain inversion does (Newton from the previous primitives is the
// fallback and decides), and *fellback is set.
template <bool SEEDED = false>
__device__ __forceinline__ int invert_zone(const Dims& d, const Params& P, const double* __restrict__ U,
                                           const double* __restrict__ pg, double* __restrict__ pf,
                                           int32_t* __restrict__ pflag, const double* __restrict__ gcent, long o,
                                           long pp, int& ns, double wp_seed = 0.0, int* fellback = nullptr)
{
  const long nc = d.ncell;
  Geom G;
  double pz[HARM_NPR];
  bool solved;
  int fl;
#pragma unroll 1
  for (int pass = 0;; pass++) {
    const double *Ur = pass ? hd::fresh(U) : U, *pgr = pass ? hd::fresh(pg) : pg;
    hd::load_geom(pass ? hd::fresh(gcent) : gcent, pp, d.nplane, G);
    double Uz[HARM_NPR];
#pragma unroll
    for (int pl = 0; pl < HARM_NPR; pl++) {
      Uz[pl] = Ur[pl * nc + o];
      pz[pl] = pgr[pl * nc + o];  // guess: the substep's starting primitives
    }
    fl = hd::utoprimgen(Uz, G, P.gam, P.gammafail, pz, ns, SEEDED && !pass ? wp_seed : __builtin_nan(""), 200, &solved);
    if (!SEEDED || pass || fl == 0) break;
    *fellback = 1;
  }
  if (!solved) {  // the guess stands (read again rather than kept through the iterations)
    const double* pgr = hd::fresh(pg);
#pragma unroll
    for (int pl = 0; pl <= HARM_U3; pl++) pz[pl] = pgr[pl * nc + o];
  }
  if (hd::needs_after_hot(fl, P.hot2cold, P.checkinv)) {
    // The rare checks and retries read the state and the geometry again,
    // through pointers the compiler cannot see through, rather than keeping
    // 70 registers through the Newton iterations (they come from L1/L2).
    hd::load_geom(hd::fresh(gcent), pp, d.nplane, G);
    double Ur[HARM_NPR], Ugf[HARM_NPR], p0[HARM_NPR];
#pragma unroll
    for (int pl = 0; pl < HARM_NPR; pl++) {
      Ur[pl] = U[pl * nc + o];
      p0[pl] = pg[pl * nc + o];
    }
    hd::geometry_free(Ur, G, Ugf);
    fl = hd::after_hot(fl, Ugf, G, P.gam, P.gammafail, p0, pz, ns, P.hot2cold, P.checkinv);
  }
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) pf[pl * nc + o] = pz[pl];
  pflag[o] = fl;
  return fl;
}

// Block sums of the Newton strokes and failures into di (integer sums are
// order independent), and the failed zones into the list behind it (room for
// `cap` zones, gkern.h; 0: no list).  Every thread of the block calls it.
__device__ __forceinline__ void newton_counts_to(int ns, int nf, unsigned long long* __restrict__ di, int zone, int cap)
{
  __shared__ unsigned long long red[2];
  if (threadIdx.x == 0) { red[0] = 0; red[1] = 0; }
  __syncthreads();
  if (ns) atomicAdd(&red[0], (unsigned long long)ns);
  if (nf) {
    atomicAdd(&red[1], 1ull);
    if (cap) {
      const unsigned long long at = atomicAdd(&di[DI_FIX], 1ull);
      if (at < (unsigned long long)cap) ((int32_t*)(di + DI_N))[at] = zone;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (red[0]) atomicAdd(&di[DI_NSTROKE], red[0]);
    if (red[1]) {
      atomicAdd(&di[DI_NFAIL], red[1]);
      if (!cap) atomicAdd(&di[DI_FIX], red[1]);
    }
  }
}

}  // namespace hk
