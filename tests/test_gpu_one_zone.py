"""Grids of a single zone: no faces, no ghosts, only the source terms and the
inversion.  A batch of them equals single grids bit for bit (its face launch had
no blocks and failed), and both are the oracle's steps."""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from harm_harm_amd.batch import Batch
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recon", ["para", "weno5"])
def test_batch_of_single_zones(recon):
    cfg = H.default_config(1, 1, 1, recon=recon, flux="hll", timeorder=2)
    og = _oracle.OGrid(cfg)
    p = og.zeros()
    p[...] = [1.0, 0.02, 0.01, 0.0, 0.02, 0.01, 0.0, 0.01]
    B, s = Batch([cfg, cfg]), Grid(cfg)
    for g in B.grids + [s]:
        g.set("p", p)
        g.set_time(0.0, 1e-3)
    B.step(5)
    s.step(5)
    for g in B.grids:
        assert np.array_equal(g.get("p"), s.get("p")) and np.array_equal(g.pflag(), s.pflag())
        assert g.newton_stats() == s.newton_stats() and g.time() == s.time()
    st, dt = og.new_state(p.copy()), 1e-3
    for _ in range(5):
        dt = og.step(st, dt)
    assert np.array_equal(s.pflag(), st["pflag"])
    assert np.allclose(s.get("p"), st["p"], rtol=1e-12, atol=0)
