"""The network's BF16 tanh (mlp.h, tanh4) against FP64's at the arguments that
decide its short form: those whose tanh lies 3 to 40 units of FP32's last place
from a point where BF16 rounding turns, on both sides of every such point from
2^-10 to 1, on both sides of the line between its two formulas (1/4), random
ones, tiny ones and saturated ones.  (Closer than 2.5 units tanhf decides, whose
own error is of that size.)

With W2 = 0 the second layer is tanh of its biases, and integer weights behind it
make an output that is exact in FP32: the sum over 64 results of one binade, 8 + 6
+ 6 bits.  One result off by a unit of BF16 changes it."""
import numpy as np
import pytest

import harm_harm_amd as H
from harm_harm_amd.mlp import MLP, NNORM, NPARAM, unpack

pytestmark = pytest.mark.gpu


def to_bf16(t):
    """FP64 to the nearest BF16 (ties to even), as FP64."""
    m, e = np.frexp(t)
    return np.ldexp(np.rint(np.ldexp(m, 8)), e - 8)


def arguments():
    rng = np.random.default_rng(1)
    x = []
    for e in range(-10, 0):
        edge = (np.arange(128, 256) + 0.5) * 2.0 ** (e - 7)
        ulp = 2.0 ** (e - 23)
        for k in (3, 4, 5, 6, 8, 10, 11, 12, 13, 14, 16, 24, 40):
            for s in (-1, 1):
                x.append(np.arctanh(edge + s * k * ulp))
    x.append(np.nextafter(np.float32(0.25), np.float32([0, 1])).astype(float))
    x.append(rng.uniform(0.24, 0.26, 2000))
    x.append(10.0 ** rng.uniform(-37, 1, 4000))
    x.append(np.array([3.5, 9.0, 20.0, 44.0, 89.0, 1e10, np.inf]))
    x = np.concatenate(x).astype(np.float32)
    x = x[np.tanh(x.astype(float)) >= 2.0**-120]
    x *= rng.choice(np.float32([-1, 1]), x.size)
    t = np.tanh(x.astype(float))
    m, e = np.frexp(np.abs(t))
    from_edge = np.abs(np.ldexp(m, 8) % 1.0 - 0.5) * 2.0**16  # in units of FP32's last place
    keep = from_edge >= 2.5
    return x[keep], to_bf16(t[keep])


def test_bf16_tanh_rounds_as_fp64s():
    x, want = arguments()
    assert x.size > 30000
    net = MLP()
    norm = np.zeros(NNORM, np.float32)
    norm[8:16] = 1.0
    norm[18:20] = 1.0
    X = H.DeviceArray.from_numpy(np.zeros((1, 8), np.float32))
    order = np.argsort(np.frexp(np.abs(want))[1], kind="stable")
    binade = np.frexp(np.abs(want))[1]
    weight = np.arange(1, 65, dtype=np.float64)
    checked = 0
    for b in np.unique(binade):
        idx = order[binade[order] == b]
        for c in range(0, idx.size, 64):
            k = idx[c:c + 64]
            w = np.zeros(NPARAM, np.float32)
            u = unpack(w)
            u["b2"][:k.size] = x[k]
            u["W3"][:k.size, 0] = weight[:k.size]
            u["W3"][:k.size, 1] = 1.0
            net.set_params(w, norm)
            y = net.forward(X, 1)
            got = y.numpy()[0]
            y.free()
            assert got[0] == np.sum(want[k] * weight[:k.size]) and got[1] == np.sum(want[k]), (b, x[k], want[k])
            checked += k.size
    assert checked == x.size
