"""The training launch at its edges: parameters and moments live in registers
for a launch and loss sums are formed every 16 steps, so launches of 1, 15, 16,
17 or 33 steps must add up to one long launch bit for bit; sample orders shorter
than a minibatch wrap; and the forward pass of a ragged number of samples gives
each sample what a full batch gives it."""
import ctypes

import numpy as np
import pytest

import harm_harm_amd as H
from harm_harm_amd.mlp import BATCH, MLP

pytestmark = pytest.mark.gpu

N = 4096


def pairs():
    rng = np.random.default_rng(3)
    X = rng.normal(size=(N, 8)).astype(np.float32) * 2
    T = np.stack([np.sin(X[:, 0]) + 0.3 * X[:, 1], np.cos(X[:, 2]) * X[:, 3]], 1).astype(np.float32)
    return [H.DeviceArray.from_numpy(a) for a in (X, T, np.ones(N, np.int32))]


def launches(dX, dT, dok, order, pieces):
    m = MLP(seed=4)
    m.fit_norm(dX, dT, dok, N)
    done, total = 0, 0.0
    for k in pieces:
        loss = ctypes.c_float()
        H.check(H.lib().harm_mlp_train(m.h, dX.ptr, dT.ptr, N, order.ptr, order.shape[0], done * BATCH, k,
                                       ctypes.c_float(2e-3), ctypes.byref(loss), None), "harm_mlp_train")
        done += k
        total += k * loss.value
    return m.params()[0], total / done


@pytest.mark.parametrize("norder", [1, 100, 128, 129, 3000])
def test_launches_add_up(norder):
    dX, dT, dok = pairs()
    order = H.DeviceArray.from_numpy(np.random.default_rng(6).permutation(N).astype(np.int32)[:norder])
    pieces = [1, 15, 16, 17, 33]
    w1, l1 = launches(dX, dT, dok, order, [sum(pieces)])
    w2, l2 = launches(dX, dT, dok, order, pieces)
    assert np.isfinite(w1).all() and np.array_equal(w1, w2)
    # the same 82 losses, averaged in float32 in another grouping
    assert abs(l1 - l2) <= 200 * 2.0**-24 * abs(l1)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 1000])
def test_forward_of_ragged_counts(n):
    dX, dT, dok = pairs()
    m = MLP(seed=4)
    m.fit_norm(dX, dT, dok, N)
    full = m.forward(dX, N).numpy()
    assert np.array_equal(m.forward(dX, n).numpy(), full[:n])
