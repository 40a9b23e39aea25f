"""2-D steps with failed zones on grids whose averaging takes several runs of
zones an item (300 x 290: 340 runs, two an item): the same bits as the separate
entry points, again and again, and no slower than they are one after the other,
each with its own launches over the whole chip and a synchronisation (with the
averaging in one block a step took several times as long)."""
import time

import numpy as np
import pytest

import harm_harm_amd as H
from harm_harm_amd.batch import Batch
from harm_harm_amd.grid import Grid
from test_gpu_bounds_launch import kicked

pytestmark = pytest.mark.gpu


def test_large_grid_with_failures_equals_kernel_sequence_and_is_no_slower():
    cfg = H.default_config(300, 290, 1, recon="para", flux="laxf", timeorder=2)
    og, p, dt = kicked(cfg, 2)
    ga, gb = Grid(cfg), Grid(cfg)
    m, CUf, Cunew = og.rk_tables()
    whole, parts = [], []
    for turn in range(6):
        for g in (ga, gb):
            g.set("p", p)
            g.set_time(0.0, dt)
            g.sync()
        t0 = time.perf_counter()
        ga.step(1)
        ga.sync()
        t1 = time.perf_counter()
        failed = 0
        for to in range(m):
            pb, pf = ("p", "pk0") if to == 0 else ("pk0", "p")
            gb.fluxcalc(pb, do_ct=True)
            gb.update("p", pb, CUf[to], Cunew[to], dt, to)
            failed += gb.invert(pb, pf, int(to == m - 1))[1]
            gb.bound(pf)
            gb.post_fixup(pf, finalstep=(to == m - 1))
            gb.bound(pf)
        gb.sync()
        whole.append(t1 - t0)
        parts.append(time.perf_counter() - t1)
        assert failed > 1000 and ga.newton_stats()[0][1] == failed
        assert np.array_equal(ga.get("p"), gb.get("p")) and np.array_equal(ga.pflag(), gb.pflag())
    assert min(whole) <= 1.2 * min(parts), (whole, parts)


def test_batch_whose_launch_exceeds_the_chip():
    """24 members of 160 x 160 zones, all but every fourth with failures: 600
    blocks where the chip holds about 512, so members' blocks start while others
    wait.  Equal to single grids over three steps."""
    cfg = H.default_config(160, 160, 1, recon="para", flux="hll", timeorder=2)
    states = []
    for seed in range(4):
        og, p, dt = kicked(cfg, seed)
        states.append((og.init_torus(), 0.3 * dt) if seed == 3 else (p, dt))
    B, singles = Batch([cfg] * 24), [Grid(cfg) for _ in states]
    for i, g in enumerate(B.grids + singles):
        p, dt = states[i % 4]
        g.set("p", p)
        g.set_time(0.0, dt)
    for step in range(3):
        B.step(1)
        for s in singles:
            s.step(1)
        want = [(s.get("p"), s.pflag(), s.newton_stats(), s.time()) for s in singles]
        for i, g in enumerate(B.grids):
            p, f, n, t = want[i % 4]
            assert np.array_equal(g.get("p"), p) and np.array_equal(g.pflag(), f), (step, i)
            assert g.newton_stats() == n and g.time() == t
    assert all(s.newton_stats()[1][1] > 0 for s in singles[:3])
