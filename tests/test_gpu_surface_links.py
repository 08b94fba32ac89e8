"""Surface force and flux from the step kernel's slots, against the CPU oracle
bit for bit: every template, after even and odd steps, bodies whose surface
links meet the faces of the block (inlets, outlets, walls, in two execution
orders), resting and turning bodies."""
import numpy as np
import pytest

from asl_amd import _lib, geometry
from gpu_common import add_bc, pair, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("steps", [1, 4, 7])
@pytest.mark.parametrize("body", ["inside", "corner", "turning"])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_force_and_flux_links(q, steps, body, dtype):
    size = (14, 11, 12)
    rng = np.random.default_rng(q + steps)
    # map nodes are counted from the ghost layer: node 1 is the first interior cell
    centre = {"inside": (6.5, 5.0, 5.5), "corner": (1.0, 1.5, 10.0), "turning": (6.5, 5.0, 5.5)}[body]
    mapv = geometry.normalize(geometry.sphere(size, 3.0, centre))
    if body == "corner":  # the outer layer is open, as ASL's drivers leave it
        outer = np.ones(mapv.shape, dtype=bool)
        outer[1:-1, 1:-1, 1:-1] = False
        mapv = np.where(outer, np.float32(1.0), mapv)
    G, O = pair(size, q, nu=0.06, dtype=dtype)
    u = (0.02 * rng.standard_normal((3,) + G.S)).astype(G.host_dtype)
    G.init_equilibrium(1.0, u)
    O.init_f(1.0, u.astype(np.float64))
    bcs = [add_bc(G, O, _lib.BC_CONSTANT_VELOCITY, _lib.X0, u=(0.03, 0.0, 0.01)),
           add_bc(G, O, _lib.BC_CONSTANT_PRESSURE_VELOCITY, _lib.ZE, p=1.01, u=(0.01, 0.0, 0.0)),
           add_bc(G, O, _lib.BC_NOSLIP, _lib.XE | _lib.Y0 | _lib.YE | _lib.Z0)]
    if body == "turning":
        bcs.append(add_bc(G, O, _lib.BC_VELOCITY_MAP, mapv=mapv, rot=(0.0, 0.0, 0.01) + centre))
    else:
        bcs.append(add_bc(G, O, _lib.BC_NOSLIP_MAP, mapv=mapv))
    if steps == 4:
        bcs = bcs[::-1]
    run(G, O, steps, bcs)
    # a link between a body cell and the outer layer (the corner body has some) exchanges what ASL's pool memory
    # holds there, which no lattice defines: cells one layer further in have none
    inner = ((slice(2, -2) if body == "corner" else slice(1, -1)),) * 3
    fg, fo = G.surface_force(mapv), O.surface_force(mapv)
    qg, qo = G.surface_flux(mapv), O.surface_flux(mapv)
    assert np.abs(np.asarray(fo)[(slice(None),) + inner]).max() > 0
    assert np.array_equal(fg[(slice(None),) + inner], np.asarray(fo)[(slice(None),) + inner].astype(G.host_dtype))
    assert np.array_equal(qg[inner], np.asarray(qo)[inner].astype(G.host_dtype))
