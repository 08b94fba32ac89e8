"""Automatic lattice groups: batches over the Infinity Cache's 256 MiB.

A batch of lattices that share groups, fill one, or exceed the cache by
themselves ends bit for bit where it ends with one group, eager and in graphs,
for few and many steps, with and without written rho and u.
"""
import numpy as np
import pytest

import asl_amd
from asl_amd import _lib
from test_gpu_batch import cavity, interior

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(108, 8, 108, 108, 40), (155, 20, 150, 9), (155, 156)])
def test_automatic_groups_equal_one_group(sizes):
    assert sum(19 * 4 * (n + 2) * (n + 3) * (n + 4) for n in sizes) > 256 << 20
    auto, one = ([cavity(n, 0.6 + 0.01 * i) for i, n in enumerate(sizes)] for _ in range(2))
    A, B = asl_amd.Batch(auto), asl_amd.Batch(one)
    B.set_tuning(_lib.TUNE_GROUP_MB, 0)
    for steps, graph, macro in ((2, False, True), (1, False, True), (9, False, False), (205, True, False), (8, True, True)):
        for batch in (A, B):
            batch.step(steps, graph=graph, write_macro=macro)
    for L, R in zip(auto, one):
        assert np.array_equal(interior(L.f()), interior(R.f()))
        assert np.array_equal(interior(L.rho()), interior(R.rho()))
        assert np.array_equal(interior(L.velocity()), interior(R.velocity()))


def test_automatic_groups_of_fp64_d3q27():
    """D3Q27 FP64 periodic lattices of 300 MiB in groups, with 256 lanes."""
    def lattices():
        out = []
        for i, n in enumerate((60, 64, 20, 70, 63, 64)):
            L = asl_amd.Lattice((n, n, n + 1), 27, dtype="f64", periodic=True, nu=0.01 * (i + 1))
            rng = np.random.default_rng(i)
            L.init_equilibrium(1.0, 0.02 * rng.standard_normal((3,) + L.S))
            out.append(L)
        return out
    auto, one = lattices(), lattices()
    A, B = asl_amd.Batch(auto), asl_amd.Batch(one)
    B.set_tuning(_lib.TUNE_GROUP_MB, 0)
    B.set_tuning(_lib.TUNE_BLOCK, 512)
    for steps, graph in ((9, False), (101, True)):
        for batch in (A, B):
            batch.step(steps, graph=graph)
    for L, R in zip(auto, one):
        assert np.array_equal(interior(L.f()), interior(R.f()))
        assert np.array_equal(interior(L.velocity()), interior(R.velocity()))
