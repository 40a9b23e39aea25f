"""WENO5BND face fluxes where the reconstruction leaves the range of its
unscaled quotients: a variable whose values are so small that the squares in
its smoothness indicators underflow takes the plain divisions, one that is
exactly zero the uniform weights, and a line whose values cross the range
mixes them zone by zone.  The oracle's divisions are IEEE, so the fluxes agree
to the per-zone bound of the step tests (they are the same operations).
"""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from _parity import assert_zones_close
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


def decayed(shape, lo, rng):
    """field values whose magnitude falls from 1e-3 to 10^lo across the box in each direction, with zeros among them"""
    e = sum(np.linspace(0.0, 1.0, n).reshape([-1 if m == a else 1 for m in range(3)]) for a, n in enumerate(shape)) / 3
    b = 10.0 ** (-3.0 + e * (lo + 3.0)) * rng.uniform(0.2, 1.0, shape) * rng.choice([-1.0, 1.0], shape)
    b[rng.uniform(size=shape) < 0.1] = 0.0
    return b


@pytest.mark.parametrize("lo", [-60, -130, -200, -320])
@pytest.mark.parametrize("n", [(20, 16, 8), (17, 21, 1)])
def test_fluxes_with_decayed_fields(n, lo):
    cfg = H.default_config(*n, recon="weno5", flux="hll", timeorder=3)
    og, g = _oracle.OGrid(cfg), Grid(cfg)
    rng = np.random.default_rng(abs(lo))
    p = og.init_torus()
    for v in (3, 4, 5, 6, 7):  # two velocity components and the field
        p[..., v] = decayed(p.shape[:3], lo, rng)
    g.set("p", p)
    F = [og.zeros() for _ in range(3)]
    ndt_o = og.fluxcalc(p, *F, do_ct=True)
    ndt_g = g.fluxcalc("p", do_ct=True)
    for d in (1, 2, 3):
        if n[d - 1] == 1:
            continue
        e = [int(d == a) for a in (3, 2, 1)]
        cut = tuple(slice(G, G + m + x) for G, m, x in zip((og.ng3, og.ng2, og.ng1), n[::-1], e))
        assert_zones_close(g.get(f"F{d}")[cut], F[d - 1][cut], f"F{d} lo {lo}")
        assert abs(ndt_g[d - 1] - ndt_o[d - 1]) <= 1e-12 * abs(ndt_o[d - 1])
