"""Divisions by the density through one reciprocal, against the CPU oracle.

The FP32 collision forms x / rho with the correctly rounded 1 / rho and a
remainder where every lane of a wavefront has a density and a momentum of
ordinary size, and divides elsewhere; both give the division's bits.  The
cases lie on either side of the line and across it: densities from 2^-30 to
2^30 within one wavefront, densities beside 2^-16 and 2^16, momenta whose
squares underflow or exceed 2^40, a resting fluid.
"""
import numpy as np
import pytest

from gpu_common import pair, run

pytestmark = pytest.mark.gpu


def fields(S, case, rng):
    z = rng.standard_normal((3,) + S)
    one = np.ones(S)
    if case == "rest":
        return one, 0.0 * z
    if case == "tiny":  # squares of 1e-38 .. 0
        return one, z * 10.0 ** rng.uniform(-30, -15, S)
    if case == "edge":
        return 2.0 ** rng.choice([-16.0, 16.0], S) * (1.0 + 2.0 ** -20 * rng.integers(-2, 3, S)), 0.02 * z
    if case == "fast":
        return one, z * 10.0 ** rng.uniform(3, 8, S)
    return 2.0 ** rng.uniform(-30, 30, S), 0.02 * z


@pytest.mark.parametrize("case", ["rest", "tiny", "edge", "fast", "spread"])
@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("turbulence", [False, True])
def test_quotients_have_the_bits_of_divisions(case, q, turbulence):
    G, O = pair((9, 8, 20), q, nu=0.05, periodic=True)
    if turbulence:
        G.set_turbulence(True)
        O.set_turbulence(True)
    rho, u = (a.astype(np.float32) for a in fields(G.S, case, np.random.default_rng(q)))
    G.init_equilibrium(rho, u)
    O.init_f(rho.astype(np.float64), u.astype(np.float64))
    run(G, O, 2, [])
    inner = (slice(1, -1),) * 3
    for g, o in ((G.f(), O.f()), (G.rho(), O.rho()), (G.velocity(), O.velocity())):
        s = (slice(None),) * (g.ndim - 3) + inner
        assert np.array_equal(g[s], np.asarray(o)[s].astype(np.float32), equal_nan=True)
