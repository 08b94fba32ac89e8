"""Sweeps (several steps of a window of planes before the next window) end
bit for bit where one launch per step ends: templates, storage types, periodic
and not, obstacles, relaxation variants, step counts around the sweep length,
eager and under graph replay, the macroscopic fields of the last step."""
import numpy as np
import pytest

import asl_amd
from asl_amd import _lib, geometry

pytestmark = pytest.mark.gpu


def build(q, dtype, periodic, variant, sweep_kb, size=(40, 7, 9)):
    L = asl_amd.Lattice(size, q, dtype=dtype, periodic=periodic, nu=0.03)
    L.set_tuning(_lib.TUNE_SWEEP_KB, sweep_kb)
    rng = np.random.default_rng(q)
    L.init_equilibrium(1.0, (0.03 * rng.standard_normal((3,) + L.S)).astype(L.host_dtype))
    if variant == "turbulence":
        L.set_turbulence(True)
    if variant == "closure":
        L.set_closure((0.1 * rng.standard_normal(_lib.CLOSURE_NPARAM)).astype(np.float32), None,
                      np.full(7, 50.0, np.float32), 0.01)
    if not periodic:
        body = geometry.normalize(geometry.sphere(size, 2.0, (18.0, 3.0, 4.0)))
        for b in (L.add_slice_bc(_lib.BC_CONSTANT_VELOCITY, _lib.X0, u=(0.03, 0, 0)),
                  L.add_slice_bc(_lib.BC_CONSTANT_PRESSURE, _lib.XE, p=1.0),
                  L.add_slice_bc(_lib.BC_NOSLIP, _lib.Y0 | _lib.YE | _lib.Z0 | _lib.ZE),
                  L.add_map_bc(_lib.BC_NOSLIP_MAP, body)):
            L.execute_bc(b)
    return L


def plane_kb(L):
    return -(-L.q * {_lib.F32: 4, _lib.F64: 8}.get(L.dtype, 2) * L.S[1] * L.S[2] // 1024)


@pytest.mark.parametrize("q,dtype,periodic,variant", [
    (19, "f32", False, None), (19, "f32", True, None), (15, "f64", False, None), (27, "f32", True, None),
    (27, "f16", False, None), (19, "bf16", True, None), (19, "f32", False, "turbulence"),
    (19, "f32", True, "closure"), (19, "f16", False, "closure")])
def test_sweeps_keep_results(q, dtype, periodic, variant):
    E = build(q, dtype, periodic, variant, 0)
    for planes in (4, 11, 30):  # 2, about 5, and 16 steps per sweep
        G = build(q, dtype, periodic, variant, plane_kb(E) * planes)
        E = build(q, dtype, periodic, variant, 0)
        for n, graph in ((1, False), (2, False), (33, False), (5, True), (16, True), (37, False)):
            G.step(n, graph=graph)
            E.step(n)
            assert np.array_equal(G.f(), E.f(), equal_nan=True), (planes, n)
            assert np.array_equal(G.rho(), E.rho()) and np.array_equal(G.velocity(), E.velocity()), (planes, n)


def test_sweep_knob():
    L = asl_amd.Lattice((6, 5, 4), 19, nu=0.1)
    assert L.tuning_value(_lib.TUNE_SWEEP_KB) == -1
    L.set_tuning(_lib.TUNE_SWEEP_KB, 64)
    assert L.tuning_value(_lib.TUNE_SWEEP_KB) == 64
    with pytest.raises(asl_amd.ASLError):
        L.set_tuning(_lib.TUNE_SWEEP_KB, -2)


@pytest.mark.parametrize("size,q,periodic", [((230, 200, 172), 19, False), ((230, 120, 130), 27, True)])
def test_automatic_sweeps_keep_results(size, q, periodic):
    """Large lattices: run lengths around the shortest ones that sweep (4; 6
    where single steps run tiles)."""
    G, E = (build(q, "f32", periodic, None, kb, size) for kb in (-1, 0))
    assert G.tuning_value(_lib.TUNE_LDS) == (0 if periodic else 1)
    for n, graph in ((3, False), (4, False), (6, False), (5, True), (19, True)):
        G.step(n, graph=graph)
        E.step(n, graph=graph)
    inner = (Ellipsis,) + (slice(1, -1),) * 3
    assert np.array_equal(G.rho()[inner], E.rho()[inner])
    assert np.array_equal(G.f()[inner], E.f()[inner])
