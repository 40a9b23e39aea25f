"""harm_set_array / harm_get_array through the handle's pinned slots: arrays of
a few kilobytes (one slot, partly filled), of just over one slot, and of more
slots than there are, so that each is used again; pageable and pinned arrays of
the caller's; two handles from two threads.  Every value must come back."""
import threading

import numpy as np
import pytest
import torch

import harm_harm_amd as H
from harm_harm_amd.grid import Grid

pytestmark = pytest.mark.gpu


def roundtrip(g, seed, pinned=False):
    shape = g.get("p").shape
    src = np.random.default_rng(seed).standard_normal(shape)
    if pinned:
        a, b = torch.empty(shape, dtype=torch.float64, pin_memory=True), torch.empty(shape, dtype=torch.float64,
                                                                                      pin_memory=True)
        a, b = a.numpy(), b.numpy()
        a[...] = src
    else:
        a, b = src.copy(), np.full(shape, np.nan)
    L = H.lib()
    H.check(L.harm_set_array(g.h, H.ARR["p"], a.ctypes.data), "set")
    H.check(L.harm_get_array(g.h, H.ARR["p"], b.ctypes.data), "get")
    assert np.array_equal(b, src)


# storage cells are 8 more a side in active directions: 0.05, 16.8, 70 and 85 MB
@pytest.mark.parametrize("n", [(16, 12, 1), (128, 24, 52), (120, 120, 60), (128, 128, 64)])
@pytest.mark.parametrize("pinned", [False, True])
def test_arrays_come_back(n, pinned):
    g = Grid(H.default_config(*n, recon="para", flux="hll", timeorder=2))
    for seed in range(3):
        roundtrip(g, seed, pinned)


def test_two_handles_from_two_threads():
    errors = []

    def work(seed):
        try:
            g = Grid(H.default_config(96, 64, 48, recon="para", flux="hll", timeorder=2))
            for k in range(4):
                roundtrip(g, 10 * seed + k)
        except BaseException as e:  # noqa: B902 - reported by the main thread
            errors.append(e)

    th = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors
