"""The matrix-core closure with its parameters in LDS: every workgroup size
(one wavefront, which copies them in several rounds, to 16) ends at the same
bits, with a last wavefront that is partly empty."""
import numpy as np
import pytest

import asl_amd
from asl_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,periodic", [("f32", True), ("f32", False), ("f16", True)])
@pytest.mark.parametrize("size", [(3, 5, 7), (9, 13, 33)])
def test_workgroup_sizes(size, dtype, periodic):
    ends = []
    for block in (512, 64, 192, 1024):
        rng = np.random.default_rng(5)
        L = asl_amd.Lattice(size, 19, dtype=dtype, periodic=periodic, nu=0.01)
        L.set_tuning(_lib.TUNE_BLOCK, block)
        L.init_equilibrium(1.0, (0.03 * rng.standard_normal((3,) + L.S)).astype(L.host_dtype))
        L.set_closure((0.2 * rng.standard_normal(_lib.CLOSURE_NPARAM)).astype(np.float32), None,
                      np.full(7, 40.0, np.float32), 0.02)
        if not periodic:
            L.execute_bc(L.add_slice_bc(_lib.BC_NOSLIP, 63))
        L.step(5)
        ends.append((L.f()[:, 1:-1, 1:-1, 1:-1].copy(), L.velocity()[:, 1:-1, 1:-1, 1:-1].copy()))
    assert np.isfinite(ends[0][0]).all()
    for f, u in ends[1:]:
        assert np.array_equal(f, ends[0][0]) and np.array_equal(u, ends[0][1])
