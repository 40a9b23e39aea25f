"""The one-launch boundary pass and the end of a substep built on it.

The pass is compared with the oracle's three directions one after the other at
the sizes its blocks change shape: one chunk of rows and several, chunk edges,
the fewest zones it takes (n1 = 8, n2 = 5, n3 = 8) and the sizes just below,
which take the direction-by-direction launches; the ghosts start scrambled, so
every one must be rebuilt.  Steps whose inversions fail (a tenth of the zones
kicked, a time step twice the Courant limit) run the parts that are skipped
otherwise: the second pass, failure averaging, in 2-D in the block that ends
last.  They are bit for bit the sequence of the separate entry points, whose
passes are unconditional, and a batch's members equal single grids.
"""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from _parity import PRIM_POSITIVE, assert_zones_close
from harm_harm_amd.batch import Batch
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


def act(og, a):
    return a[og.ng3:og.ng3 + og.cfg.n3, og.ng2:og.ng2 + og.cfg.n2, og.ng1:og.ng1 + og.cfg.n1]


@pytest.mark.parametrize("n", [(8, 5, 1), (7, 5, 1), (9, 63, 1), (12, 64, 1), (10, 65, 1), (33, 130, 1), (8, 5, 8),
                               (7, 9, 8), (9, 32, 8), (11, 33, 10), (20, 70, 8), (12, 6, 12)])
def test_bounds_match_oracle(n):
    cfg = H.default_config(*n, recon="para", flux="laxf", timeorder=2)
    og, g = _oracle.OGrid(cfg), Grid(cfg)
    p = og.zeros()
    rng = np.random.default_rng(sum(n))
    p[...] = rng.uniform(-3.0, 3.0, p.shape)
    a = act(og, p)
    a[..., 0:2] = rng.uniform(0.1, 1.0, a.shape[:3] + (2,))
    a[..., 2:8] = 0.1 * rng.normal(size=a.shape[:3] + (6,))
    g.set("p", p)
    g.bound("p")
    og.bound(p)
    assert_zones_close(g.get("p"), p, f"bound {n}", positive=PRIM_POSITIVE)


def kicked(cfg, seed):
    """A torus with a tenth of its zones kicked out of the inversion's reach, and a time step twice the limit."""
    og = _oracle.OGrid(cfg)
    p = og.init_torus()
    a = act(og, p)
    rng = np.random.default_rng(seed)
    m = rng.uniform(size=a.shape[:3]) < 0.1
    a[m, 2:5] += 2.0 * rng.normal(size=(m.sum(), 3)) * [1.0, 0.05, 0.05]
    a[m, 5:8] += 0.02 * rng.normal(size=(m.sum(), 3))
    og.bound(p)
    ndt = og.fluxcalc(p, og.zeros(), og.zeros(), og.zeros())
    return og, p, 2.0 * min(x for x in ndt if x < 1e50)


CASES = [((24, 20, 1), "para", 2), ((40, 70, 1), "para", 3), ((33, 66, 1), "weno5", 2), ((16, 12, 8), "para", 2),
         ((18, 34, 10), "weno5", 3), ((16, 4, 8), "para", 2), ((7, 12, 1), "para", 2)]


@pytest.mark.parametrize("n,recon,rk", CASES)
def test_step_with_failures_equals_kernel_sequence(n, recon, rk):
    cfg = H.default_config(*n, recon=recon, flux="laxf", timeorder=rk)
    og, p, dt = kicked(cfg, 2)
    ga, gb = Grid(cfg), Grid(cfg)
    for g in (ga, gb):
        g.set("p", p)
    ga.set_time(0.0, dt)
    m, CUf, Cunew = og.rk_tables()
    pbb = ["p", "pk0", "pk1"] if m == 3 else ["p", "pk0"]
    pff = ["pk0", "pk1", "p"] if m == 3 else ["pk0", "p"]
    for step in range(3):
        failed = 0
        dts = ga.time()[1]
        ga.step(1)
        for to in range(m):
            gb.fluxcalc(pbb[to], do_ct=True)
            gb.update("p", pbb[to], CUf[to], Cunew[to], dts, to)
            failed += gb.invert(pbb[to], pff[to], int(to == m - 1))[1]
            gb.bound(pff[to])
            gb.post_fixup(pff[to], finalstep=(to == m - 1))
            gb.bound(pff[to])
        assert np.array_equal(ga.get("p"), gb.get("p")), step
        assert np.array_equal(ga.pflag(), gb.pflag()), step
        assert ga.newton_stats()[0][1] == failed
        assert step > 0 or failed > 0  # the first step fails somewhere


@pytest.mark.parametrize("ns", [[(24, 20, 1), (40, 70, 1), (64, 33, 1)], [(16, 12, 8), (18, 34, 10)]])
def test_batch_with_failures_equals_single_grids(ns):
    cfgs = [H.default_config(*n, recon="para", flux="hll", timeorder=2) for n in ns]
    B = Batch(cfgs)
    singles = [Grid(c) for c in cfgs]
    for i, c in enumerate(cfgs):
        og, p, dt = kicked(c, 3 + i)
        if i == 1:
            p, dt = og.init_torus(), 0.3 * dt  # one member without failures
        for g in (B.grids[i], singles[i]):
            g.set("p", p)
            g.set_time(0.0, dt)
    for step in range(3):
        B.step(1)
        for g, s in zip(B.grids, singles):
            s.step(1)
            assert np.array_equal(g.get("p"), s.get("p")) and np.array_equal(g.pflag(), s.pflag())
            assert g.newton_stats() == s.newton_stats() and g.time() == s.time()
    assert singles[0].newton_stats()[1][1] > 0
