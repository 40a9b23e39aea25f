"""The batched inversion's split of a call into rounds: up to 262144 zones each
run of 256 is a block of its own; beyond that a block takes several runs, stops
their solves early and solves the unfinished zones again in full waves.  The
zones are independent, so a call gives every zone the bits, flag and iteration
count that calls on parts of at most 100000 zones give it; the sample holds
zones of 6 to 200 iterations (those that circle until the cap among them),
failed hot solves with their cold retry and failed zones.
"""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from harm_harm_amd.sampling import sample_inversion_inputs

pytestmark = pytest.mark.gpu


def sample(n):
    p, guess, geom = sample_inversion_inputs(min(n, 1 << 16), seed=21)
    r = -(-n // p.shape[1])
    p, guess, geom = (np.ascontiguousarray(np.tile(a, (1, r))[:, :n]) for a in (p, guess, geom))
    U = _oracle.p2u_batch(p, geom)
    rng = np.random.default_rng(5)
    bad = rng.integers(0, n, max(1, n // 50))
    U[1, bad] = np.abs(U[1, bad]) * 3.0
    U[0, rng.integers(0, n, max(1, n // 200))] *= -1.0
    return U, geom, guess


def invert(U, geom, guess):
    D = H.DeviceArray
    n = U.shape[1]
    dU, dg, dq = D.from_numpy(U), D.from_numpy(geom), D.from_numpy(guess)
    fl, it = D.zeros(n, np.int32), D.zeros(n, np.int32)
    H.check(H.lib().harm_invert_batch(dU.ptr, dg.ptr, dq.ptr, fl.ptr, it.ptr, n, 4.0 / 3.0, 2500.0, None), "invert")
    H.synchronize()
    return dq.numpy(), fl.numpy(), it.numpy()


@pytest.mark.parametrize("n", [1, 255, 257, 262144, 262145, 300001, 700000])
def test_rounds_equal_parts(n):
    U, geom, guess = sample(n)
    p, fl, it = invert(U, geom, guess)
    for c in range(0, n, 100000):
        s = slice(c, min(n, c + 100000))
        q, f, i = invert(*(np.ascontiguousarray(a[:, s]) for a in (U, geom, guess)))
        assert np.array_equal(p[:, s], q) and np.array_equal(fl[s], f) and np.array_equal(it[s], i)
    m = min(n, 1 << 16)
    po, fo, io = _oracle.invert_batch(U[:, :m], geom[:, :m], guess[:, :m])
    assert np.array_equal(fl[:m], fo) and np.array_equal(it[:m], io)
    assert np.max(np.abs(p[:, :m] - po) / np.maximum(np.abs(po), 1e-300)) <= 1e-12
    assert n < 1000 or ((it == 200).any() and (fl > 0).any())  # the sample holds what it should
