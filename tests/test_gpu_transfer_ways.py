"""Host transfers each way and size that takes a way of its own (one buffer up
to 2 MiB to the host, the ring from there; the runtime's path below 14 MiB to the
device), from and into ordinary and pinned memory: every byte comes back."""
import ctypes

import numpy as np
import pytest
import torch

import asl_amd
from asl_amd import _lib

pytestmark = pytest.mark.gpu


# a view is 76 (nx + 2) (ny + 2) (nz + 2) bytes: 2 kB, just below and above 2 MiB and 14 MiB, 48 MB
@pytest.mark.parametrize("size", [(1, 1, 1), (20, 41, 27), (22, 21, 48), (44, 66, 59), (44, 68, 59), (70, 90, 94)])
@pytest.mark.parametrize("pinned_in", [False, True])
@pytest.mark.parametrize("pinned_out", [False, True])
def test_views_come_back(size, pinned_in, pinned_out):
    L = asl_amd.Lattice(size, 19, periodic=True, nu=0.1)
    n = 19 * L.len
    rng = np.random.default_rng(n)
    a = torch.empty(n, dtype=torch.float32, pin_memory=pinned_in)
    b = torch.empty(n, dtype=torch.float32, pin_memory=pinned_out)
    a.numpy()[:] = rng.integers(-1000, 1000, n)
    b.fill_(7)
    for _ in range(2):
        _lib.call("aslhip_write_f", L.h, ctypes.c_void_p(a.data_ptr()))
        a.numpy()[:] += 1  # the lattice has its copy by now
        _lib.call("aslhip_read_f", L.h, ctypes.c_void_p(b.data_ptr()))
        assert np.array_equal(b.numpy(), a.numpy() - 1)
