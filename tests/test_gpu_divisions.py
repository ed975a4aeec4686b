"""The kernels' own division and square root: velocities and fluxes over a wide
range of magnitudes.  Velocities are correctly rounded quotients, so they equal
numpy's bit for bit, and so does the pressure (no fused operations); the flux's
square roots and reciprocals round as before, and it is held to the reference
formula in numpy's float64 with the bound of the pointwise tests."""
import numpy as np
import pytest

from fvs2d_amd import meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("decades", [1, 30, 100])
def test_primitives_are_correctly_rounded(decades):
    m = meshgen.jittered_square(70, periodic=True, seed=1)
    s = Solver(m, vortex_scheme(dt=0.01))
    rng = np.random.default_rng(decades)
    mag = lambda: 10.0 ** rng.uniform(-decades, decades, s.ncells)  # noqa: E731
    u = np.stack([mag(), mag() * rng.choice([-1.0, 1.0], s.ncells), -mag(), mag()], 1)
    u[::7, 1] = 0.0
    s.cvar = u
    w = s.cvar2pvar()
    v1, v2 = u[:, 1] / u[:, 0], u[:, 2] / u[:, 0]
    assert np.array_equal(w[:, 0], u[:, 0]) and np.array_equal(w[:, 1], v1) and np.array_equal(w[:, 2], v2)
    assert np.array_equal(w[:, 3], (1.4 - 1.0) * (u[:, 3] - 0.5 * u[:, 0] * (v1 * v1 + v2 * v2)))


@pytest.mark.parametrize("bad", [0.0, np.nan, np.inf])
def test_impossible_density_stays_visible(bad):
    m = meshgen.jittered_square(12, periodic=True, seed=1)
    s = Solver(m, vortex_scheme(dt=0.01, limiter=1))
    s.initialize_solution(1, 0.0)
    u = s.cvar
    u[5, 0] = bad
    s.cvar = u
    assert not np.all(np.isfinite(s.cvar2pvar()[5]))
    r, _ = s.compute_residual(0.0)
    assert not np.all(np.isfinite(r[5]))
