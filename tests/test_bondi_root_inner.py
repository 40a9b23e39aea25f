"""The Newton root of the Bondi boundary in the innermost band that ghost zones
may lie in, 0.35 < r < 0.5, where f' mostly lies outside the range that Newton
accepts and the reference's iteration decides: the few roots that are accepted
(of boundary zones far from the flow's integrals) are the iteration's."""
import ctypes
import math

import numpy as np
import pytest

from test_bondi_root import iterate, newton  # noqa: F401


@pytest.mark.parametrize("wide,least", [(0.02, 0), (0.6, 20)])
def test_accepted_roots_are_the_iterations(newton, wide, least):  # noqa: F811
    rng = np.random.default_rng(5)
    taken = 0
    for _ in range(12000):
        gam, rs, r = rng.uniform(1.2, 1.65), rng.uniform(5.5, 20.0), rng.uniform(0.35, 0.5)
        n = 1 / (gam - 1)
        us = math.sqrt(1 / (2 * rs))
        V2 = us * us / (1 - 3 * us * us)
        Ts = -n * V2 / ((n + 1) * (n * V2 - 1))
        C1 = us * rs * rs * Ts**n * rng.uniform(1 - wide, 1 + wide)
        C2 = (1 + (1 + n) * Ts) ** 2 * (1 - 2 / rs + us * us) * rng.uniform(1 - wide, 1 + wide)
        ref, settled = iterate(n, C1, C2, r)
        start = (ref if settled and ref > 0 else Ts) * rng.uniform(1 - wide, 1 + wide)
        T = ctypes.c_double(start)
        if newton(n, C1, C2, r, ctypes.byref(T)):
            taken += 1
            assert settled and abs(T.value - ref) <= 1e-12 * abs(ref), (n, C1, C2, r, start)
    assert taken >= least
