"""Host copies through the pinned ring: sizes around a chunk (2 MiB), around
the ring (16 MiB) and where threads come in, several threads at once, the ring
given back and taken again."""
import threading

import numpy as np
import pytest

import asl_amd

pytestmark = pytest.mark.gpu


def round_trip(size, seed, q=19, dtype="f32"):
    L = asl_amd.Lattice(size, q, dtype=dtype, periodic=True, nu=0.1)
    f = np.random.default_rng(seed).standard_normal((q,) + L.S).astype(L.host_dtype)
    L.write_f(f)
    return np.array_equal(L.f(), f)


# one view is Q (nx + 2) (ny + 2) (nz + 2) values: from 11 kB through 2 MiB and 16 MiB and their neighbours to 47 MB
@pytest.mark.parametrize("size", [(3, 4, 3), (10, 10, 47), (15, 43, 39), (17, 42, 31), (29, 41, 40), (30, 64, 104),
                                  (31, 64, 103), (70, 90, 94)])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_views_come_back(size, dtype):
    assert round_trip(size, 1, dtype=dtype)


def test_many_threads():
    """Transfers of several threads, one of which has the ring at a time."""
    ok = []

    def work(k):
        ok.append(all(round_trip((20 + 5 * k, 40, 50), 10 * k + i) for i in range(4)))
    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert ok == [True] * 6


def test_ring_is_given_back_and_taken_again():
    for k in range(3):
        assert round_trip((8, 30, 40), k)  # the only lattice of its time
