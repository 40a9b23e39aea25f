"""Grids without an x2 direction: radial lines and (r, phi) planes, alone and in
a batch.  They have no polar rows, so their boundary pass is the radial
extrapolation and the phi copies only (test_bounds_plan.py walks the merged
pass's blocks for the sizes it takes).  Ghosts start scrambled in the boundary
test; whole steps compare primitives and dt with the oracle's to 1e-12 a zone
and the flags exactly; a batch's members equal single grids bit for bit (a batch
of grids whose dimensions differ is refused)."""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from _parity import PRIM_POSITIVE, assert_zones_close
from harm_harm_amd.batch import Batch
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu

SIZES = [(7, 1, 1), (8, 1, 1), (33, 1, 1), (300, 1, 1), (7, 1, 8), (16, 1, 8), (33, 1, 12)]


def start(cfg, seed):
    """A perturbed torus, or the Bondi flow, and a third of its time step."""
    og = _oracle.OGrid(cfg)
    if cfg.problem == 1:
        p = og.init_bondi()
    else:
        p = og.init_torus()
        a = p[og.ng3:og.ng3 + cfg.n3, :, og.ng1:og.ng1 + cfg.n1]
        a[...] *= 1.0 + 0.02 * np.random.default_rng(seed).uniform(-1, 1, a.shape)
        og.bound(p)
    ndt = og.fluxcalc(p, og.zeros(), og.zeros(), og.zeros())
    return og, p, 0.3 * min(x for x in ndt if x < 1e50)


def configs():
    for n in SIZES:
        yield H.default_config(*n, recon="para", flux="laxf", timeorder=2)
    yield H.default_config(33, 1, 12, recon="weno5", flux="hll", timeorder=3)
    yield H.default_config(64, 1, 1, recon="weno5", flux="laxf", timeorder=2)
    yield H.bondi_config(64, 1, recon="para", flux="laxf", timeorder=2)


@pytest.mark.parametrize("cfg", list(configs()), ids=lambda c: f"{c.problem}-{c.n1}-{c.n3}-{c.recon}")
def test_radial_grid_matches_oracle(cfg):
    og, p, dt = start(cfg, 2)
    g = Grid(cfg)
    q = np.random.default_rng(4).uniform(-3.0, 3.0, p.shape)
    s = np.s_[og.ng3:og.ng3 + cfg.n3, :, og.ng1:og.ng1 + cfg.n1]
    q[s] = p[s]
    g.set("p", q)
    g.bound("p")
    og.bound(q)
    assert_zones_close(g.get("p"), q, "bound", positive=PRIM_POSITIVE)
    g.set("p", p)
    g.set_time(0.0, dt)
    st = og.new_state(p.copy())
    for step in range(5):  # a graph of four and one of one
        dt = og.step(st, dt)
    g.step(5)
    assert_zones_close(g.get("p")[s], st["p"][s], "step", positive=PRIM_POSITIVE)
    assert np.array_equal(g.pflag(), st["pflag"])
    assert abs(g.time()[1] - dt) <= 1e-12 * dt


@pytest.mark.parametrize("ns", [[(16, 1, 1), (7, 1, 1), (100, 1, 1)], [(16, 1, 8), (33, 1, 12)]])
def test_batch_of_radial_grids_equals_single_grids(ns):
    cfgs = [H.default_config(*n, recon="para", flux="hll", timeorder=2) for n in ns]
    B = Batch(cfgs)
    singles = [Grid(c) for c in cfgs]
    for i, c in enumerate(cfgs):
        og, p, dt = start(c, 3 + i)
        for g in (B.grids[i], singles[i]):
            g.set("p", p)
            g.set_time(0.0, dt)
    B.step(5)
    for g, s in zip(B.grids, singles):
        s.step(5)
        assert np.array_equal(g.get("p"), s.get("p")) and np.array_equal(g.pflag(), s.pflag())
        assert g.newton_stats() == s.newton_stats() and g.time() == s.time()


def test_mixed_dimensions_are_refused():
    with pytest.raises(H.HarmError, match="dimensionality"):
        Batch([H.default_config(*n, recon="para", flux="hll", timeorder=2) for n in [(40, 1, 1), (24, 20, 1)]])
