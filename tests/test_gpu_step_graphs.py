"""Steps replayed as graphs of one and of four: a call of n steps gives the bits
of n calls of one, for counts around the longer graph's length, with host work
and the energy sums switched on and off (which captures again) in between."""
import numpy as np
import pytest

import harm_harm_amd as H
from harm_harm_amd.batch import Batch
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


def start(n, recon, rk):
    g = Grid(H.default_config(*n, recon=recon, flux="hll", timeorder=rk))
    g.init_torus(seed=4)
    ndt = [x for x, m in zip(g.fluxcalc("p"), n) if m > 1]
    g.set_time(0.0, 0.5 / sum(1.0 / x for x in ndt))
    return g


def state(g):
    return [g.get("p"), g.get("ucum"), g.pflag(), np.array(g.time()), np.array(g.newton_stats())]


@pytest.mark.parametrize("n,recon,rk", [((24, 20, 1), "para", 2), ((20, 16, 8), "weno5", 3)])
def test_calls_add_up(n, recon, rk):
    a, b = start(n, recon, rk), start(n, recon, rk)
    for count in (1, 3, 4, 5, 8, 11):
        a.step(count)
        for _ in range(count):
            b.step(1)
        if count == 5:  # other kernels from here on, and back
            a.set_ener_tracking(True)
            b.set_ener_tracking(True)
        if count == 8:
            a.set_ener_tracking(False)
            b.set_ener_tracking(False)
        for x, y in zip(state(a), state(b)):
            assert np.array_equal(x, y)


def test_batch_calls_add_up():
    cfgs = [H.default_config(24, 20, 1, recon="para", flux="laxf", timeorder=2),
            H.bondi_config(32, 16, recon="para", flux="laxf", timeorder=2)]
    runs = []
    for whole in (True, False):
        B = Batch(cfgs)
        for g in B.grids:
            g.init_bondi() if g is B.grids[1] else g.init_torus(seed=4)
            ndt = g.fluxcalc("p")[:2]
            g.set_time(0.0, 0.5 / sum(1.0 / x for x in ndt))
        for count in (3, 4, 9):
            for _ in range(1 if whole else count):
                B.step(count if whole else 1)
        runs.append([(g.get("p"), np.array(g.time())) for g in B.grids])
    for (p, t), (q, u) in zip(*runs):
        assert np.array_equal(p, q) and np.array_equal(t, u)
