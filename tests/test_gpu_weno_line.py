"""The WENO5BND line pass with a zone a thread (grids of up to about 400 000
zones) against the oracle at the sizes its blocks change shape: one segment a
line and two, the longest line of one segment (118 zones, with 120 faces), the
shortest lines, column tiles that end inside the face box; and the sweep on a
grid just large enough for it.
"""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from _parity import assert_zones_close
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(8, 5, 8), (11, 119, 1), (13, 120, 1), (12, 121, 1), (9, 250, 1), (14, 7, 118),
                               (10, 6, 122), (64, 4, 10), (112, 52, 64), (129, 65, 66), (141, 64, 64)])
def test_fluxes_match_oracle(n):
    cfg = H.default_config(*n, recon="weno5", flux="laxf", timeorder=2)
    og, g = _oracle.OGrid(cfg), Grid(cfg)
    rng = np.random.default_rng(n[1])
    p = og.zeros()
    p[..., 0:2] = rng.uniform(0.1, 1.0, p.shape[:3] + (2,))
    p[..., 2:8] = 0.1 * rng.normal(size=p.shape[:3] + (6,))
    # half of the box smooth, so that SMONO, WENO5 and the reduced weights all occur
    x = np.arange(p.shape[2])[None, None, :, None] + 0.3 * np.arange(p.shape[1])[None, :, None, None]
    h = p.shape[1] // 2
    p[:, :h] = (0.5 + 0.3 * np.sin(0.2 * x + np.arange(8)))[:, :h]
    F = [og.zeros() for _ in range(3)]
    ndt_o = og.fluxcalc(p, *F, do_ct=True)
    g.set("p", p)
    ndt_g = g.fluxcalc("p", do_ct=True)
    for d in (1, 2, 3):
        if n[d - 1] == 1:
            continue
        e = [int(d == a) for a in (3, 2, 1)]
        cut = tuple(slice(G, G + m + x) for G, m, x in zip((og.ng3, og.ng2, og.ng1), n[::-1], e))
        assert_zones_close(g.get(f"F{d}")[cut], F[d - 1][cut], f"{n} F{d}")
        assert abs(ndt_g[d - 1] - ndt_o[d - 1]) <= 1e-12 * abs(ndt_o[d - 1])
