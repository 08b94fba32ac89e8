"""The sweeps' launch order at the limits of its arguments, on the CPU: the
launches of the definition (block b of g planes does planes [b g - s, (b + 1) g -
s) in step s, those that exist), numbers near 2^31, refusals."""
import ctypes

import numpy as np
import pytest

from asl_amd import _lib
from test_sweep_plan import plan

BIG = 2**31 - 1


def definition(nx, periodic, g, t, n):
    out = []
    for s0 in range(0, n, t):
        m = min(t, n - s0)
        b = 0
        while b * g - (m - 1) < (nx + m - 1 if periodic else nx):
            for s in range(m):
                lo, hi = max(b * g - s, s if periodic else 0), min((b + 1) * g - s, nx + s if periodic else nx)
                if lo < hi and lo < nx:
                    out.append((s0 + s, lo, min(hi, nx) - lo))
                if lo < hi and hi > nx:
                    out.append((s0 + s, max(lo, nx) - nx, hi - max(lo, nx)))
            b += 1
    return out


@pytest.mark.parametrize("periodic", [False, True])
def test_launches_of_the_definition(periodic):
    rng = np.random.default_rng(1)
    for _ in range(300):
        nx, g, t, n = (int(rng.integers(1, k)) for k in (40, 30, 20, 50))
        t = min(t, nx)
        assert [tuple(r) for r in plan(nx, periodic, g, t, n)] == definition(nx, periodic, g, t, n), (nx, g, t, n)


def test_large_arguments():
    for periodic in (False, True):
        assert [tuple(r) for r in plan(BIG, periodic, 2**30, 2, 3)] == definition(BIG, periodic, 2**30, 2, 3)
        assert len(plan(BIG, periodic, BIG, 3, 3)) == len(definition(BIG, periodic, BIG, 3, 3))
    lib = _lib.load_library()
    assert lib.aslhip_sweep_plan(BIG, 0, 1, 1, 2, None, 0) < 0  # more launches than an int counts
    assert lib.aslhip_sweep_plan(5, 1, 2, 6, 6, None, 0) < 0  # a ring of 5 planes cannot be 6 steps ahead of itself
    one = np.full(9, -1, dtype=np.int32)
    assert lib.aslhip_sweep_plan(20, 0, 5, 3, 3, one.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), 1) > 1
    assert list(one[:4]) == [0, 0, 5, -1]
