"""Gradient and training of the closure network where the kernels' blocks end:
batches around 32 samples (a column block), 128 (a workgroup), 32768 (from one
to two blocks per wavefront), ranges that start inside the data, against FP64.

Tolerance: an entry is a sum over samples of products of FP32 values that are
themselves chains of at most 7 + 32 + 32 + 32 fused operations; with at most
64 samples per FP32 partial sum that is under 200 roundings of 2^-24, 1.2e-5 of
the largest terms at worst.

The gradient jumps where a unit's input changes sign.  A unit whose FP64 input
is nearer to zero than FP32 can tell (40000 samples hold one, at 1.4e-8) may be
on in one arithmetic and off in the other, so the reference is the gradient
with either choice for such units.
"""
import numpy as np
import pytest

import asl_amd
from oracle import mlp

pytestmark = pytest.mark.gpu


def gradient_beside(g, p, x, t):
    """The FP64 gradient, with the choice nearest to g for each unit that FP32 cannot decide."""
    W1, b1, W2, b2, w3, b3 = mlp.unpack(p)
    y, (a1, h1, a2, h2) = mlp.forward(p, x)
    u = 2.0 ** -24
    near1 = np.abs(a1) < 8 * u * (np.abs(x) @ np.abs(W1).T + np.abs(b1))
    near2 = np.abs(a2) < 33 * u * (np.abs(h1) @ np.abs(W2).T + np.abs(b2))
    unsure = [(1, i) for i in np.argwhere(near1)] + [(2, i) for i in np.argwhere(near2)]
    # a choice moves the gradient by that sample's share alone
    dy = (y - t) / len(x)
    base = mlp.loss_and_grad(p, x, t)[1]

    def share(layer, i):
        g = np.zeros_like(base)
        on2 = a2[i[0]] > 0
        if layer == 2:
            k, sign = i[1], -1.0 if on2[i[1]] else 1.0
            d2 = np.zeros(mlp.H)
            d2[k] = sign * dy[i[0]] * w3[k]
            d1 = (d2 @ W2) * (a1[i[0]] > 0)
        else:
            d2 = np.zeros(mlp.H)
            d1 = np.zeros(mlp.H)
            d1[i[1]] = (-1.0 if a1[i[0], i[1]] > 0 else 1.0) * ((dy[i[0]] * w3 * on2) @ W2)[i[1]]
        g[:224] = np.outer(d1, x[i[0]]).ravel()
        g[224:256] = d1
        g[256:1280] = np.outer(d2, h1[i[0]]).ravel()
        g[1280:1312] = d2
        return g
    assert len(unsure) <= 1e-3 * len(x)
    for layer, i in unsure:
        d = share(layer, i)
        if np.abs(g - base - d).max() < np.abs(g - base).max():
            base = base + d
    return base


@pytest.mark.parametrize("first,count", [(0, 1), (3, 31), (0, 32), (5, 33), (0, 127), (1, 128), (0, 129), (0, 255),
                                         (7, 257), (0, 32768), (0, 32769), (11, 40000)])
def test_gradient_at_block_edges(first, count):
    rng = np.random.default_rng(count)
    x = rng.standard_normal((first + count + 2, 7)).astype(np.float32)
    t = (x[:, 0] * x[:, 1] + rng.standard_normal(len(x))).astype(np.float32)
    p = mlp.init_params(3)
    m = asl_amd.Mlp(p)
    m.set_data(x, t)
    loss, g = m.gradient(first, count)
    lr, _ = mlp.loss_and_grad(p.astype(np.float64), x[first:first + count], t[first:first + count])
    assert abs(loss - lr) <= 1.2e-5 * lr
    gr = gradient_beside(g, p.astype(np.float64), x[first:first + count].astype(np.float64), t[first:first + count])
    assert np.abs(g - gr).max() <= 1.2e-5 * np.abs(gr).max()
    again = m.gradient(first, count)
    assert again[0] == loss and np.array_equal(again[1], g)


def test_losses_of_long_runs_arrive_in_order():
    """A run longer than one copy of the losses (4096 steps) equals the same
    steps in short runs, and the losses are those of the steps."""
    rng = np.random.default_rng(0)
    x = rng.standard_normal((500, 7)).astype(np.float32)
    t = x[:, 0].astype(np.float32)
    a, b = (asl_amd.Mlp(mlp.init_params(4)) for _ in range(2))
    for m in (a, b):
        m.set_data(x, t)
    la = a.train(4100, 64, 1e-3, 7)
    lb = np.concatenate([b.train(n, 64, 1e-3, 7) for n in (1, 2000, 2099)])
    assert np.array_equal(la, lb) and np.array_equal(a.params(), b.params())
