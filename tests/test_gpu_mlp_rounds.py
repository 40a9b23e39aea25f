"""The seeded batched inversion's rounds: up to 196608 zones each run of 256 is a
block of its own, beyond that a block takes several runs, and zones whose seeded
solve is unfinished or has failed are solved again in full waves.  The zones
are independent, so a call gives every zone the bits, flag and iteration count
that calls on parts of at most 100000 zones give it, and the fallbacks add up.
Seeds far off (a network that answers a constant) make most zones unfinished or
failed; where a zone fell back, its flag is the plain inversion's.
"""
import numpy as np
import pytest

import _oracle
import harm_harm_amd as H
from harm_harm_amd.mlp import MLP, NPARAM
from harm_harm_amd.sampling import sample_inversion_inputs

pytestmark = pytest.mark.gpu

D = H.DeviceArray


def sample(n):
    p, guess, geom = sample_inversion_inputs(min(n, 1 << 16), seed=22)
    r = -(-n // p.shape[1])
    p, guess, geom = (np.ascontiguousarray(np.tile(a, (1, r))[:, :n]) for a in (p, guess, geom))
    U = _oracle.p2u_batch(p, geom)
    bad = np.random.default_rng(6).integers(0, n, max(1, n // 50))
    U[1, bad] = np.abs(U[1, bad]) * 3.0
    return U, geom, guess


def invert(m, U, geom, guess):
    n = U.shape[1]
    dU, dg, dq = D.from_numpy(U), D.from_numpy(geom), D.from_numpy(guess)
    fl, it, fb = D.zeros(n, np.int32), D.zeros(n, np.int32), D.zeros(1, np.uint64)
    if m is None:
        H.check(H.lib().harm_invert_batch(dU.ptr, dg.ptr, dq.ptr, fl.ptr, it.ptr, n, 4.0 / 3.0, 2500.0, None), "inv")
    else:
        m.invert_batch(dU, dg, dq, fl, it, n, dfallback=fb)
    H.synchronize()
    return dq.numpy(), fl.numpy(), it.numpy(), int(fb.numpy()[0])


@pytest.mark.parametrize("n", [1, 255, 257, 196608, 196609, 300001])
@pytest.mark.parametrize("bias", [0.0, 40.0])  # log(W'/D) of the constant answer
def test_rounds_equal_parts(n, bias):
    m = MLP(seed=1)
    w = np.zeros(NPARAM, np.float32)
    w[-2] = bias
    m.set_params(w=w)
    U, geom, guess = sample(n)
    p, fl, it, fb = invert(m, U, geom, guess)
    fbs = 0
    for c in range(0, n, 100000):
        s = slice(c, min(n, c + 100000))
        q, f, i, b = invert(m, *(np.ascontiguousarray(a[:, s]) for a in (U, geom, guess)))
        assert np.array_equal(p[:, s], q) and np.array_equal(fl[s], f) and np.array_equal(it[s], i)
        fbs += b
    assert fb == fbs
    pq, fq, iq, _ = invert(None, U, geom, guess)
    print(n, bias, "fallbacks", fb, "plain mean", iq.mean(), "seeded", it.mean(), "failed", (fq > 0).sum(), (fl > 0).sum())
    # a zone whose seeded solve fails is decided by the plain one, so none fails that the plain one solves
    assert not ((fl != 0) & (fq == 0)).any()
    assert n < 1000 or fb > 0
