"""The direct step kernel's items and face rule, against the CPU oracle.

Workgroups take consecutive interior cells whatever the rows and planes they
belong to, so the sizes here put row and plane ends inside wavefronts and
chunks: rows of one cell, planes of one row, chunks over many planes, a last
chunk of one cell.  Every face has a boundary condition of its own, with and
without values, in two execution orders (which decides the edge links).
Same operations in the same order on both sides: bit for bit.
"""
import numpy as np
import pytest

from asl_amd import _lib
from gpu_common import add_bc, compare, pair, run

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 1, 67), (70, 3, 1), (1, 300, 2), (5, 3, 129), (13, 9, 7), (4, 33, 64)]


def six_faces(G, O, rng):
    kinds = [(_lib.BC_CONSTANT_VELOCITY, dict(u=(0.02, 0.01, -0.01))), (_lib.BC_CONSTANT_PRESSURE, dict(p=1.01)),
             (_lib.BC_NOSLIP, {}), (_lib.BC_CONSTANT_PRESSURE_VELOCITY, dict(p=0.99, u=(0.01, -0.02, 0.0))),
             (_lib.BC_NOSLIP, {}), (_lib.BC_CONSTANT_VELOCITY, dict(u=(-0.01, 0.02, 0.0)))]
    faces = [_lib.X0, _lib.XE, _lib.Y0, _lib.YE, _lib.Z0, _lib.ZE]
    kinds = [kinds[i] for i in rng.permutation(6)]
    bcs = [add_bc(G, O, k, f, **p) for (k, p), f in zip(kinds, faces)]
    return [bcs[i] for i in rng.permutation(6)]


@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("wide", [0, 1])
def test_rows_planes_and_faces(size, q, wide):
    rng = np.random.default_rng(q + sum(size))
    for dtype, block in (("f32", 512), ("f64", 64)):
        G, O = pair(size, q, nu=0.08, dtype=dtype)
        G.set_tuning(_lib.TUNE_WIDE, wide)
        G.set_tuning(_lib.TUNE_BLOCK, block)
        u = 0.02 * rng.standard_normal((3,) + G.S)
        u = u.astype(G.host_dtype)
        G.init_equilibrium(1.0, u)
        O.init_f(1.0, u.astype(np.float64))
        run(G, O, 7, six_faces(G, O, rng))
        d = compare(G, O)
        assert d["rho"] == 0.0 and d["u"] == 0.0 and d["f"] == 0.0, (dtype, d)


@pytest.mark.parametrize("size", [(3, 3, 3), (2, 5, 66), (40, 3, 4)])
@pytest.mark.parametrize("q", [19, 27])
def test_periodic_wrap(size, q):
    rng = np.random.default_rng(sum(size))
    for dtype in ("f32", "f64"):
        G, O = pair(size, q, nu=0.05, dtype=dtype, periodic=True)
        u = (0.02 * rng.standard_normal((3,) + G.S)).astype(G.host_dtype)
        G.init_equilibrium(1.0, u)
        O.init_f(1.0, u.astype(np.float64))
        run(G, O, 6, [])
        d = compare(G, O)
        assert d["rho"] == 0.0 and d["u"] == 0.0 and d["f"] == 0.0, (dtype, d)


@pytest.mark.parametrize("size", [(1, 1, 1), (2, 3, 1), (1, 2, 65), (9, 1, 3), (7, 8, 9)])
@pytest.mark.parametrize("q", [15, 19, 27])
def test_conservation_wraps_after_odd_steps(size, q):
    """Sums after 1 to 3 steps: the wrap along axes of one, two and more cells.
    FP64 sums of the same terms in another order differ by less than
    (number of terms) x 2^-53 of the sum of their magnitudes."""
    rng = np.random.default_rng(q + sum(size))
    for dtype, periodic in (("f32", True), ("f64", True), ("f64", False)):
        G, O = pair(size, q, nu=0.08, dtype=dtype, periodic=periodic)
        u = (0.02 * rng.standard_normal((3,) + G.S)).astype(np.float32)
        G.init_equilibrium(1.0, u)
        O.init_f(1.0, u.astype(np.float64))
        bcs = [] if periodic else six_faces(G, O, rng)
        run(G, O, 0, bcs)
        mask = np.zeros(G.S, dtype=np.uint8)
        mask[1:-1, 1:-1, 1:-1] = 1
        n = int(np.prod(size))
        for _ in range(3):
            G.step(1)
            O.run(1, [o for _, o in bcs])
            tol = 4 * q * n * 2.0**-53 * n * 2  # |w c f| summed: at most 2 per cell
            assert np.abs(np.subtract(G.conservation(), O.conservation(mask))).max() <= tol


@pytest.mark.parametrize("size", [(1, 1, 5), (32, 32, 32), (33, 32, 32), (64, 32, 32), (65, 32, 32)])
def test_small_lattices_pick_their_workgroup(size):
    """Without a choice of the caller's, lattices around the limits of 32768
    and 65536 cells end bit for bit where 512-lane workgroups take them."""
    for q, dtype, periodic in ((19, "f32", False), (27, "f64", True), (15, "f32", False)):
        ends = []
        for block in (None, 512):
            rng = np.random.default_rng(q)
            G, O = pair(size, q, nu=0.08, dtype=dtype, periodic=periodic)
            if block:
                G.set_tuning(_lib.TUNE_BLOCK, block)
            G.init_equilibrium(1.0, (0.02 * rng.standard_normal((3,) + G.S)).astype(np.float32))
            run(G, O, 0, [] if periodic else six_faces(G, O, rng))
            G.step(3)
            G.step(205, graph=True)
            assert G.tuning()[0] == 512
            ends.append((G.f(), G.rho(), G.velocity()))
        inner = (Ellipsis,) + (slice(1, -1),) * 3
        assert all(np.array_equal(a[inner], b[inner], equal_nan=True) for a, b in zip(*ends))


@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("compressible", [True, False])
def test_turbulence_in_a_rotating_frame(q, dtype, compressible):
    """LBGKTurbulence forms the equilibria once, and again after the frame's
    term; GPU vs oracle bit for bit, the frame switched on after plain steps."""
    size = (9, 7, 11)
    rng = np.random.default_rng(q)
    S = tuple(s + 2 for s in size)
    f0 = 1.0 + rng.uniform(0.01, 0.8, S) * rng.standard_normal((q,) + S)
    G, O = pair(size, q, nu=0.2, dtype=dtype, periodic=True, compressible=compressible)
    for L in (G, O):
        L.set_turbulence(True)
    G.write_f(f0)
    O.write_f(G.f().astype(np.float64))
    s = (slice(None),) + (slice(1, -1),) * 3
    for om in (None, (0.004, -0.002, 0.01)):
        for L in (G, O):
            L.set_omega(om)
        G.step(5)
        O.run(5)
        fo = O.f()[s].astype(G.f().dtype)
        assert np.isfinite(fo).all()
        assert np.array_equal(G.f()[s], fo)
