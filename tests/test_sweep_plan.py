"""The launch order of the sweeps (several steps of a window of planes before
the next window), checked against what a step needs, on the CPU: a plane's
step needs the plane and both neighbours one step earlier, and every plane
takes every step once."""
import ctypes

import numpy as np
import pytest

from asl_amd import _lib


def plan(nx, periodic, planes, steps, n):
    lib = _lib.load_library()
    count = lib.aslhip_sweep_plan(nx, int(periodic), planes, steps, n, None, 0)
    assert count >= 0
    out = np.zeros((max(count, 1), 3), dtype=np.int32)
    assert lib.aslhip_sweep_plan(nx, int(periodic), planes, steps, n,
                                 out.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), count) == count
    return out[:count]


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("nx", [3, 4, 7, 16, 61])
def test_every_plane_takes_every_step_after_its_neighbours(nx, periodic):
    for planes in (1, 2, 3, 8):
        for steps in (1, 2, 3, 5, 8):
            if planes + steps >= nx:  # the library sweeps windows of fewer planes than the lattice has
                continue
            for n in (0, 1, 2, steps, steps + 1, 3 * steps + 2):
                done = np.zeros(nx, dtype=int)  # steps taken by each plane
                for s, p0, k in plan(nx, periodic, planes, steps, n):
                    assert k >= 1 and p0 >= 0 and p0 + k <= nx
                    for p in range(p0, p0 + k):
                        assert done[p] == s, (planes, steps, n, s, p)
                        for d in (-1, 1):
                            q = p + d
                            if periodic:
                                q %= nx
                            elif not 0 <= q < nx:
                                continue
                            # the neighbour has taken the step before, and not this one's successor
                            assert s <= done[q] or (p0 <= q < p0 + k), (planes, steps, n, s, p, q)
                            assert done[q] <= s + 1, (planes, steps, n, s, p, q)
                    done[p0:p0 + k] = s + 1
                assert (done == n).all()


def test_bad_arguments():
    lib = _lib.load_library()
    assert lib.aslhip_sweep_plan(0, 0, 1, 1, 1, None, 0) < 0
    assert lib.aslhip_sweep_plan(4, 0, 0, 1, 1, None, 0) < 0
    assert lib.aslhip_sweep_plan(4, 0, 1, 1, 1, None, 5) < 0
