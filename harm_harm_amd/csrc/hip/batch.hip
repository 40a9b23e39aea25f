// batch.hip -- per-zone kernels over n independent zones (SoA device buffers).
//
// harm_invert_batch: Utoprimgen (utoprimgen.c:32) for the inversion
// microbench, as the torus configuration compiles it (the hot solve, then the
// cold retry of a failed one; no inversion check); harm_prim_to_cons_batch: primtoU(UEVOLVE) (phys.tools.c:475).
#include <hip/hip_runtime.h>
#include <algorithm>
#include "dphys.h"
#include "hhost.h"

namespace {

constexpr int kBlock = 256;

// Zone z's inversion with at most `limit` Newton iterations; false, with
// nothing written, when the solve needs more.
__device__ __forceinline__ bool invert_one(const double* __restrict__ U, const double* __restrict__ geom,
                                           double* __restrict__ p, int32_t* __restrict__ pflag,
                                           int32_t* __restrict__ niter, long n, double gam, double gammafail, long z,
                                           int limit)
{
  hd::Geom g;
  hd::load_geom(geom, z, n, g);
  double Uz[HARM_NPR], pz[HARM_NPR];
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) {
    Uz[pl] = U[pl * n + z];
    pz[pl] = p[pl * n + z];
  }
  int ns = 0;
  bool solved;
  int fl = hd::utoprimgen<true>(Uz, g, gam, gammafail, pz, ns, __builtin_nan(""), limit, &solved);
  if (fl == hd::kUnfinishedFlag) return false;
  if (!solved) {  // the guess stands (read again rather than kept through the iterations)
    const double* pr = hd::fresh(p);
#pragma unroll
    for (int pl = 0; pl <= HARM_U3; pl++) pz[pl] = pr[pl * n + z];
  }
  if (hd::needs_after_hot(fl, true, false)) {  // HOT2COLD (the torus configuration)
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
  return true;
}

// A block takes `rounds` runs of 256 zones.  A wave's solve lasts as long as
// its slowest zone's, and the counts differ widely: 90 % of the zones of a
// log-uniform sample take at most 18 iterations, 7 % take 50 to 56 (the
// reference halves the steps after ten), so that without further measures a
// wave's mean is 160 (counting the zones that run to the cap, newton<CYCLE>)
// for a zone's 17.5.  With more than one round the solves stop at kFirst
// iterations; the unfinished zones go into a list in LDS and are solved from
// the start, in full waves, whenever a block's worth has come together and
// after the last round.  2^24 zones take 5.5 ms (27.5 ms one zone a lane to the
// end; 7.0 GB compulsory, so 1.3 TB/s).  4096 zones take 0.09 ms, the slowest
// zone's chain of 30 to 50 iterations (its cycles are counted, not run); with the
// 200 that it has to its cap a round trip through p -> U -> p took 0.38, now 0.16.
// Compared with one another on one box: kFirst 12, 14, 16 and 18 5.9, 5.1, 4.9 and
// 4.9 ms; four waves per SIMD although 136 B a lane spill 4.9, three 5.3, two 6.0.
constexpr int kFirst = 16;
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_invert_batch(const double* __restrict__ U, const double* __restrict__ geom,
                                                         double* __restrict__ p, int32_t* __restrict__ pflag,
                                                         int32_t* __restrict__ niter, long n, double gam,
                                                         double gammafail, int rounds)
{
  const int tid = threadIdx.x;
  const long z0 = (long)blockIdx.x * kBlock * rounds;
  const int first = rounds > 1 ? kFirst : 200;
  __shared__ int list[2 * kBlock];  // zones (from z0) left unfinished, at most 255 + 256
  __shared__ int cnt;
  if (tid == 0) cnt = 0;
  __syncthreads();
  int round = 0;
#pragma clang loop unroll(disable)
  while (true) {
    const int c = __builtin_amdgcn_readfirstlane(cnt);  // the same in every thread: cnt changes between barriers only
    const bool more = round < rounds && z0 + (long)round * kBlock < n;
    if (!more && c == 0) break;
    const bool full = c >= kBlock || !more;
    int loc = -1;
    if (full) {
      const int take = min(c, kBlock);
      if (tid < take) loc = list[c - 1 - tid];
    } else {
      if (z0 + (long)round * kBlock + tid < n) loc = round * kBlock + tid;
      round++;
    }
    __syncthreads();  // the list's entries and cnt have been read
    if (full && tid == 0) cnt = c - min(c, kBlock);
    __syncthreads();
    if (loc >= 0 && !invert_one(U, geom, p, pflag, niter, n, gam, gammafail, z0 + loc, full ? 200 : first))
      list[atomicAdd(&cnt, 1)] = loc;
    __syncthreads();
  }
}

__global__ __launch_bounds__(kBlock) void k_p2u_batch(const double* __restrict__ p, const double* __restrict__ geom,
                                                      double* __restrict__ U, long n, double gam)
{
  const long z = (long)blockIdx.x * kBlock + threadIdx.x;
  if (z >= n) return;
  hd::Geom g;
  hd::load_geom(geom, z, n, g);
  double pz[HARM_NPR], Uz[HARM_NPR];
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) pz[pl] = p[pl * n + z];
  hd::State q;
  hd::get_state(pz, g, gam, q);
  hd::primtoflux(pz, q, 0, g, Uz);
#pragma unroll
  for (int pl = 0; pl < HARM_NPR; pl++) U[pl * n + z] = Uz[pl];
}

}  // namespace

extern "C" harm_status harm_invert_batch(const double* U, const double* geom, double* p_inout, int32_t* pflag,
                                         int32_t* niter, int64_t n, double gam, double gammafail, void* stream)
{
  if (n <= 0 || !U || !geom || !p_inout || !pflag) return hh::set_error(HARM_EINVAL, "invert_batch: bad arguments");
  const long nr = (long)((n + kBlock - 1) / kBlock);
  if (nr > 0x7fffffffL) return hh::set_error(HARM_EINVAL, "invert_batch: n too large");
  constexpr long kResident = 1024;  // blocks the chip holds (four waves a SIMD)
  const int rounds = hh::inversion_rounds(nr, kResident);
  const long nb = (nr + rounds - 1) / rounds;
  hipLaunchKernelGGL(k_invert_batch, dim3((unsigned)nb), dim3(kBlock), 0, (hipStream_t)stream, U, geom, p_inout, pflag,
                     niter, (long)n, gam, gammafail, rounds);
  return hh::check_launch("k_invert_batch");
}

extern "C" harm_status harm_prim_to_cons_batch(const double* p, const double* geom, double* U, int64_t n, double gam,
                                               void* stream)
{
  if (n <= 0 || !p || !geom || !U) return hh::set_error(HARM_EINVAL, "prim_to_cons_batch: bad arguments");
  const long nb = (long)((n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_p2u_batch, dim3((unsigned)nb), dim3(kBlock), 0, (hipStream_t)stream, p, geom, U, (long)n, gam);
  return hh::check_launch("k_p2u_batch");
}
