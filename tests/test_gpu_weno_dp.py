"""The dP measure's tiles: blocks of 32 x 8 zones with a halo of one march
through chunks of k planes.  Sizes that leave one zone, one short of a tile,
and whole tiles in i (30) and j (6), and chunks of two planes with a remainder;
random states whose pressure jumps pass the measure's thresholds, so that the
reduced stencils depend on it.  Fluxes agree with the oracle's to the per-zone
bound of the step tests."""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from _parity import assert_zones_close
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(28, 16, 8), (29, 17, 10), (27, 15, 12), (58, 10, 14), (59, 22, 8), (17, 21, 1), (28, 16, 1)])
def test_fluxes_over_tile_edges(n):
    cfg = H.default_config(*n, recon="weno5", flux="hll", timeorder=3)
    og, g = _oracle.OGrid(cfg), Grid(cfg)
    rng = np.random.default_rng(sum(n))
    p = og.init_torus()
    sh = p.shape[:3]
    p[..., 0] = 10.0 ** rng.uniform(-2, 0, sh)
    p[..., 1] = 10.0 ** rng.uniform(-4, -1, sh)
    for v in (2, 3, 4):
        p[..., v] = rng.uniform(-0.3, 0.3, sh) / (1.0, 10.0, 10.0)[v - 2]
    for v in (5, 6, 7):
        p[..., v] = rng.uniform(-0.05, 0.05, sh)
    g.set("p", p)
    F = [og.zeros() for _ in range(3)]
    ndt_o = og.fluxcalc(p, *F, do_ct=True)
    ndt_g = g.fluxcalc("p", do_ct=True)
    for d in (1, 2, 3):
        if n[d - 1] == 1:
            continue
        e = [int(d == a) for a in (3, 2, 1)]
        cut = tuple(slice(G, G + m + x) for G, m, x in zip((og.ng3, og.ng2, og.ng1), n[::-1], e))
        assert_zones_close(g.get(f"F{d}")[cut], F[d - 1][cut], f"F{d} n {n}")
        assert abs(ndt_g[d - 1] - ndt_o[d - 1]) <= 1e-12 * abs(ndt_o[d - 1])
