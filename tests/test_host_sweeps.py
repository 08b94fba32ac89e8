"""When runs of steps sweep by themselves, over the stand-in for the HIP runtime
(host_hip.py): a sweep is several launches a step, otherwise there is one."""
import pytest

import host_hip


@pytest.mark.parametrize("size,q,dtype,periodic,steps,sweeps", [
    # a window of 224 MiB holds fewer than 16 planes: no gain where the lattice is not large
    ((20, 400, 300), 19, "f64", True, 20, False), ((20, 400, 300), 19, "f64", False, 20, False),
    ((24, 512, 512), 19, "f32", True, 20, False), ((40, 700, 700), 27, "f32", True, 20, False),
    ((40, 500, 500), 27, "f64", True, 20, False), ((30, 750, 750), 19, "f16", True, 20, False),
    ((80, 512, 512), 19, "f32", True, 20, True), ((80, 400, 300), 19, "f64", False, 20, False),
    ((130, 400, 300), 19, "f64", False, 20, True),
    # 16 planes and more
    ((160, 150, 150), 19, "f64", True, 20, True), ((160, 150, 150), 19, "f64", True, 8, True),
    ((160, 150, 150), 19, "f64", True, 7, False), ((170, 170, 170), 27, "f16", False, 4, True),
    ((170, 170, 170), 27, "f16", False, 3, False), ((160, 150, 150), 27, "f32", True, 4, True),
    # tiles, and lattices that the cache holds
    ((256, 128, 128), 19, "f32", False, 20, False), ((128, 128, 128), 19, "f32", True, 20, False)])
def test_automatic_sweeps(size, q, dtype, periodic, steps, sweeps):
    host_hip.run("""
L = cavity(%r, %d, dtype=%r, periodic=%r)
L.step(2)
launches()
L.step(%d)
n = len(launches())
assert n > %d if %r else n == %d, n
""" % (size, q, dtype, periodic, steps, steps, sweeps, steps))
