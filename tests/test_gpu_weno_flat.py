"""WENO5BND where the five values of a window are equal (the shortcut of
zone_weights) and where all but one are: piecewise constant variables of many
magnitudes, blocks of 3 to 9 zones in each direction, so that every window
position against an edge occurs.  The oracle has no shortcut; the fluxes agree
to the per-zone bound of the step tests."""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from _parity import assert_zones_close
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [3, 5, 6, 9])
@pytest.mark.parametrize("n", [(20, 16, 8), (17, 21, 1)])
def test_fluxes_with_flat_blocks(n, block):
    cfg = H.default_config(*n, recon="weno5", flux="hll", timeorder=3)
    og, g = _oracle.OGrid(cfg), Grid(cfg)
    rng = np.random.default_rng(block)
    p = og.init_torus()
    sh = p.shape[:3]
    idx = np.ix_(*[np.arange(m) // block for m in sh])
    for v, (lo, hi) in enumerate([(-6, 0), (-8, -2), (-3, -1), (-3, -1), (-3, -1), (-200, -3), (-200, -3), (-3, -2)]):
        small = [int(x.max()) + 1 for x in idx]
        b = 10.0 ** rng.uniform(lo, hi, small)
        if v >= 2:
            b *= rng.choice([-1.0, 0.0, 1.0], small)
        p[..., v] = b[idx]
    g.set("p", p)
    F = [og.zeros() for _ in range(3)]
    ndt_o = og.fluxcalc(p, *F, do_ct=True)
    ndt_g = g.fluxcalc("p", do_ct=True)
    for d in (1, 2, 3):
        if n[d - 1] == 1:
            continue
        e = [int(d == a) for a in (3, 2, 1)]
        cut = tuple(slice(G, G + m + x) for G, m, x in zip((og.ng3, og.ng2, og.ng1), n[::-1], e))
        assert_zones_close(g.get(f"F{d}")[cut], F[d - 1][cut], f"F{d} block {block}")
        assert abs(ndt_g[d - 1] - ndt_o[d - 1]) <= 1e-12 * abs(ndt_o[d - 1])
