"""One velocity BC on several faces that meet: the links on their common edges
and corners belong to the BC once, whatever the number of its faces they enter
through.  GPU vs oracle bit for bit on every path of the step (one cell per
lane, 64-bit addresses, runs of cells, tiles, sweeps, batches, LBGKTurbulence),
the BC executed first and last, and the surface force of a body at such an edge."""
import numpy as np
import pytest

import asl_amd
from asl_amd import _lib, geometry
from gpu_common import add_bc, compare, pair

pytestmark = pytest.mark.gpu

ALL = _lib.X0 | _lib.XE | _lib.Y0 | _lib.YE | _lib.Z0 | _lib.ZE
FACES = [_lib.X0 | _lib.ZE, _lib.XE | _lib.YE, _lib.Y0 | _lib.Z0, _lib.X0 | _lib.Y0 | _lib.ZE,
         _lib.XE | _lib.YE | _lib.Z0, _lib.X0 | _lib.XE | _lib.Y0, ALL]
PATHS = {"direct": [(_lib.TUNE_LDS, 0)], "wide": [(_lib.TUNE_WIDE, 1)], "run 2": [(_lib.TUNE_CPL, 2)],
         "run 4": [(_lib.TUNE_CPL, 4)], "tiles": [(_lib.TUNE_LDS, 1)], "even tiles": [(_lib.TUNE_LDS, 2)],
         "sweeps": [(_lib.TUNE_SWEEP_KB, None)], "batch": [], "batch tiles": [], "turbulence": []}


def bcs_of(G, O, faces, kind, first):
    """The BC on `faces`, walls on the others, in that order or the other one."""
    out = [add_bc(G, O, kind, faces, p=1.01, u=(0.05, 0.01, 0.02))]
    if faces != ALL:
        out.append(add_bc(G, O, _lib.BC_NOSLIP, ALL & ~faces))
    return out if first else out[::-1]


@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_edges_and_corners(q, path, dtype):
    size = (7, 5, 8)
    for i, faces in enumerate(FACES):
        for kind in (_lib.BC_CONSTANT_VELOCITY, _lib.BC_CONSTANT_PRESSURE_VELOCITY):
            rng = np.random.default_rng(q + i)
            G, O = pair(size, q, nu=0.08, dtype=dtype)
            for knob, value in PATHS[path]:
                if value is None:  # a window of five planes
                    value = -(-5 * q * np.dtype(G.host_dtype).itemsize * G.S[1] * G.S[2] // 1024)
                G.set_tuning(knob, value)
            if path == "turbulence":
                G.set_turbulence(True)
                O.set_turbulence(True)
            u = (0.02 * rng.standard_normal((3,) + G.S)).astype(G.host_dtype)
            G.init_equilibrium(1.0, u)
            O.init_f(1.0, u.astype(np.float64))
            bcs = bcs_of(G, O, faces, kind, i % 2 == 0)
            for g, o in bcs:
                G.execute_bc(g)
                O.execute_bc(o)
            stepper = G
            if path.startswith("batch"):
                stepper = asl_amd.Batch([G])
                stepper.set_tuning(_lib.TUNE_LDS, int(path == "batch tiles"))
            stepper.step(7)
            O.run(7, [o for _, o in bcs])
            d = compare(G, O)
            assert d["rho"] == 0.0 and d["u"] == 0.0 and d["f"] == 0.0, (faces, kind, d)


@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("steps", [4, 7])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_force_of_a_body_at_the_edge(q, steps, dtype):
    size = (14, 11, 12)
    rng = np.random.default_rng(q + steps)
    # node 1 is the first interior cell: the sphere covers part of the edge between X0 and ZE
    mapv = geometry.normalize(geometry.sphere(size, 3.0, (1.0, 5.0, 11.0)))
    outer = np.ones(mapv.shape, dtype=bool)
    outer[1:-1, 1:-1, 1:-1] = False
    mapv = np.where(outer, np.float32(1.0), mapv)  # the outer layer is open, as ASL's drivers leave it
    G, O = pair(size, q, nu=0.06, dtype=dtype)
    u = (0.02 * rng.standard_normal((3,) + G.S)).astype(G.host_dtype)
    G.init_equilibrium(1.0, u)
    O.init_f(1.0, u.astype(np.float64))
    bcs = bcs_of(G, O, _lib.X0 | _lib.ZE, _lib.BC_CONSTANT_VELOCITY, True)
    bcs.append(add_bc(G, O, _lib.BC_NOSLIP_MAP, mapv=mapv))
    for g, o in bcs:
        G.execute_bc(g)
        O.execute_bc(o)
    G.step(steps)
    O.run(steps, [o for _, o in bcs])
    d = compare(G, O)
    assert d["rho"] == 0.0 and d["u"] == 0.0 and d["f"] == 0.0, d
    # links between the body and the outer layer exchange what ASL's pool memory holds there: one layer further in
    inner = (slice(None),) + (slice(2, -2),) * 3
    fg, fo = G.surface_force(mapv), np.asarray(O.surface_force(mapv))
    assert np.abs(fo[inner]).max() > 0
    assert np.array_equal(fg[inner], fo[inner].astype(G.host_dtype))
