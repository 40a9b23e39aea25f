"""The Newton root of the Bondi boundary (dgrid.h, bondi_newton) against the
reference's iterations from T = 0.1, on the host: the function's source is
compiled as C++ and called over random adiabatic indices, sonic points, radii
and perturbed boundary zones.  Where it accepts, both must be the same root.
The iterations leave an error of a few rounding units over 0.02 (f' - 1) >= 0.14
or 1 - f' >= 0.13, below 1e-14; 1e-12 is asked for."""
import ctypes
import math
import os
import re
import subprocess

import numpy as np
import pytest

HDR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "harm_harm_amd", "csrc", "hip", "dgrid.h")


@pytest.fixture(scope="module")
def newton(tmp_path_factory):
    src = re.search(r"__device__ __forceinline__ bool bondi_newton.*?\n}\n", open(HDR).read(), re.S).group(0)
    d = tmp_path_factory.mktemp("bondi")
    cc, so = str(d / "b.cc"), str(d / "b.so")
    with open(cc, "w") as f:
        f.write("#include <math.h>\n#define __device__\n#define __forceinline__ inline\n" + src)
        f.write('extern "C" int root(double n, double C1, double C2, double r, double* T)'
                "{ return bondi_newton(n, C1, C2, r, *T); }\n")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", cc, "-o", so], check=True)
    fn = ctypes.CDLL(so).root
    fn.argtypes = [ctypes.c_double] * 4 + [ctypes.POINTER(ctypes.c_double)]
    return fn


def iterate(n, C1, C2, r):
    """(T, settled): the damped iteration inside r = 2.5, the plain one outside r = 9."""
    T0, T1 = 0.2, 0.1
    try:
        for _ in range(250):
            T0 = T1
            u = C1 / (r * r * math.pow(T0, n))
            f = (math.sqrt(C2 / (1 - 2 / r + u * u)) - 1) / (1 + n)
            T1 = T0 + 0.02 * (T0 - f) if r < 2.5 else f
            rel = (T0 - T1) / T1
            if (abs(rel) if r < 2.5 else rel) <= 1e-15:
                # an outer step that rises by rounding alone has settled too
                return T1, r < 2.5 or T1 <= T0 * (1 + 1e-14)
    except (ValueError, ZeroDivisionError, OverflowError):
        pass
    return T1, False


@pytest.mark.parametrize("rlo,rhi", [(0.5, 1.5), (1.5, 2.5), (9.0, 12.0), (12.0, 60.0)])
@pytest.mark.parametrize("wide", [0.02, 0.6])
def test_newton_root_is_the_iterations_root(newton, rlo, rhi, wide):
    rng = np.random.default_rng(int(rlo * 10 + 1000 * wide))
    taken = worst = wrong = 0
    for _ in range(1500):
        gam, rs = rng.uniform(1.2, 1.65), rng.uniform(5.5, 20.0)
        r = rng.uniform(rlo, rhi)
        n = 1 / (gam - 1)
        us = math.sqrt(1 / (2 * rs))
        V2 = us * us / (1 - 3 * us * us)
        Ts = -n * V2 / ((n + 1) * (n * V2 - 1))
        if not 0 < Ts < 1:
            continue
        C1 = us * rs * rs * Ts**n * rng.uniform(1 - wide, 1 + wide)
        C2 = (1 + (1 + n) * Ts) ** 2 * (1 - 2 / rs + us * us) * rng.uniform(1 - wide, 1 + wide)
        ref, settled = iterate(n, C1, C2, r)
        start = (ref if settled and ref > 0 else Ts) * rng.uniform(1 - wide, 1 + wide)
        T = ctypes.c_double(start)
        if newton(n, C1, C2, r, ctypes.byref(T)):
            taken += 1
            if not settled:
                wrong += 1
            else:
                worst = max(worst, abs(T.value - ref) / abs(ref))
    print(rlo, rhi, wide, "taken", taken, "worst", worst, "unsettled", wrong)
    assert wrong == 0 and taken > 100
    assert worst <= 1e-12


@pytest.mark.parametrize("T", [float("nan"), float("inf"), 0.0, -0.1, 1e-300])
def test_bad_start_is_refused_or_finds_the_root(newton, T):
    n, C1, C2 = 3.0, 0.0, 1.1
    t = ctypes.c_double(T)
    assert not newton(n, C1, C2, 1.3, ctypes.byref(t))
