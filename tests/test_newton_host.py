"""The inversion's source (dphys.h) on the host, over zones that have a solution
and zones that have none, whose iterations leave the domain and go back with
half the step: flags, strokes and primitives are the oracle's, with and without
the counting of cycles, and no iteration forms the general residual more than
once (the one at the point it goes back to is kept)."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

import _oracle
from harm_harm_amd.sampling import sample_inversion_inputs

HIP = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "harm_harm_amd", "csrc", "hip")

HEAD = r"""
#include <cmath>
#include <cstdint>
#include <algorithm>
using std::isfinite;
#define __device__
#define __host__
#define __forceinline__ inline
static inline double __builtin_amdgcn_rcp(double x) { return 1.0 / x; }
static long nresidual;
"""

TAIL = r"""
template <bool CYCLE>
static void solve(const double* U, const double* geom, double* p, int32_t* fl, int32_t* ns, int32_t* nr, long n)
{
  for (long z = 0; z < n; z++) {
    hd::Geom g;
    hd::load_geom(geom, z, n, g);
    double Uz[HARM_NPR], Ugf[HARM_NPR], p0[HARM_NPR], pz[HARM_NPR];
    for (int q = 0; q < HARM_NPR; q++) {
      Uz[q] = U[q * n + z];
      pz[q] = p0[q] = p[q * n + z];
    }
    nresidual = 0;
    int s = 0, f = hd::utoprimgen<CYCLE>(Uz, g, 4.0 / 3.0, 2500.0, pz, s, __builtin_nan(""));
    if (hd::needs_after_hot(f, true, false)) {
      hd::geometry_free(Uz, g, Ugf);
      f = hd::after_hot(f, Ugf, g, 4.0 / 3.0, 2500.0, p0, pz, s, true, false);
    }
    for (int q = 0; q < HARM_NPR; q++) p[q * n + z] = pz[q];
    fl[z] = f;
    ns[z] = s;
    nr[z] = (int32_t)nresidual;
  }
}
extern "C" void run(const double* U, const double* geom, double* p, int32_t* fl, int32_t* ns, int32_t* nr, long n, int cycle)
{
  if (cycle) solve<true>(U, geom, p, fl, ns, nr, n);
  else solve<false>(U, geom, p, fl, ns, nr, n);
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    src = open(os.path.join(HIP, "dphys.h")).read().replace("#include <hip/hip_runtime.h>", "")
    src, a = re.subn(r"(double\* fresh\(const double\* p\)\n)\{.*?\n\}", r"\1{ return p; }", src, flags=re.S)
    src, b = re.subn(r"(__forceinline__ void residual\([^{]*\)\n\{)", r"\1 nresidual++;", src)
    assert a == 1 and b == 1
    d = tmp_path_factory.mktemp("newton")
    cc, so = str(d / "n.cc"), str(d / "n.so")
    with open(cc, "w") as f:
        f.write(HEAD + src + TAIL)
    inc = os.path.join(HIP, "..", "..", "..", "include")
    subprocess.run(["g++", "-O1", "-ffp-contract=off", "-std=c++17", "-shared", "-fPIC", "-I", inc, "-I", HIP, cc, "-o", so],
                   check=True)
    fn = ctypes.CDLL(so).run

    def call(U, geom, guess, cycle):
        n = U.shape[1]
        p = guess.copy()
        fl, ns, nr = (np.zeros(n, np.int32) for _ in range(3))
        fn(*(ctypes.c_void_p(x.ctypes.data) for x in (U, geom, p, fl, ns, nr)), ctypes.c_long(n), ctypes.c_int(cycle))
        return p, fl, ns, nr

    return call


@pytest.mark.parametrize("kick", ["none", "momentum", "energy", "noise"])
def test_matches_the_oracle_with_one_residual_an_iteration(run, kick):
    p, guess, geom = sample_inversion_inputs(3000, seed=11)
    U = _oracle.p2u_batch(p, geom)
    rng = np.random.default_rng(3)
    if kick == "momentum":
        U[2:5] *= rng.uniform(1.0, 3.0, (3, 3000))
    elif kick == "energy":
        U[1] *= rng.uniform(-0.5, 1.5, 3000)
    elif kick == "noise":
        U *= 1.0 + 0.5 * rng.normal(size=U.shape)
    po, fo, io = _oracle.invert_batch(U, geom, guess)
    assert kick == "none" or np.mean(fo != 0) > 0.2
    for cycle in (0, 1):
        q, fl, ns, nr = run(U, geom, guess, cycle)
        assert np.array_equal(fl, fo) and np.array_equal(ns, io)
        same = (q == po) | (np.isnan(q) & np.isnan(po))
        assert same.all(), np.argwhere(~same)[:5]
        assert np.all(nr <= ns), (nr - ns).max()
