"""Persistent whole-step launches next to the other routes of a context: meshes
whose block ranges are cut (the reference order on many cells, quadrilaterals in
the reference order) take them, and a context that changes between them and two
kernels per stage continues from its current state.  Bit for bit the kernels of
kernel_path 3."""
import numpy as np
import pytest

from fvs2d_amd import _lib, meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu


def quads(nx, ny):
    """nx x ny quadrilaterals on a sheared rectangle, periodic in both directions."""
    i, j = (a.ravel() for a in np.meshgrid(np.arange(nx + 1), np.arange(ny + 1)))
    xy = np.stack([-5 + 10 * i / nx + 0.3 * j / ny, -5 + 10 * j / ny], 1).astype(float)
    qi, qj = (a.ravel() for a in np.meshgrid(np.arange(nx), np.arange(ny)))
    bl = qj * (nx + 1) + qi
    cells = np.stack([bl, bl + 1, bl + nx + 2, bl + nx + 1], 1)
    canon = ((j % ny) * (nx + 1) + i % nx).astype(np.int32)
    return meshgen.Mesh(xy, 0, nx * ny, cells.ravel().astype(np.int32), [], canon=canon, period=(10.0, 10.0))


MESHES = {
    "many triangles": lambda: meshgen.jittered_square(132, periodic=True, seed=2),
    "quads": lambda: quads(96, 70),
}


@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("mesh", list(MESHES))
def test_reference_order_takes_persistent_launches(mesh, limiter):
    m, sch = MESHES[mesh](), vortex_scheme(dt=1e-3, limiter=limiter, reorder=0)
    a, b, c = Solver(m, sch, kernel_path=3), Solver(m, sch, kernel_path=2), Solver(m, sch, kernel_path=2)
    c.set_persistent(True)
    for s in (a, b, c):
        s.initialize_solution(1, 0.0)
    for n in (5, 4):
        na, nb, nc = (s.time_integration(0.0, n) for s in (a, b, c))
        assert np.array_equal(na, nb) and np.array_equal(na, nc)
    assert np.array_equal(a.cvar, b.cvar) and np.array_equal(a.cvar, c.cvar)


@pytest.mark.parametrize("rk", [_lib.RK_SSP3, _lib.RK_SSP42_SO, _lib.RK_SSP42])
def test_switching_routes_continues_from_the_state(rk):
    m = meshgen.jittered_square(40, periodic=True, seed=5)
    sch = vortex_scheme(dt=2e-3, reorder=1, rk_scheme=rk)
    a, b = Solver(m, sch, kernel_path=3), Solver(m, sch, kernel_path=2)
    for s in (a, b):
        s.initialize_solution(1, 0.0)
    b.set_launch_choices({"gradient": 2})
    for persistent in (False, True, False, True):
        b.set_persistent(persistent)
        na, nb = a.time_integration(0.0, 5), b.time_integration(0.0, 5)
        assert np.array_equal(na, nb) and np.array_equal(a.cvar, b.cvar)


def test_error_records_between_persistent_launches():
    """A call with vortex-error records runs single launches; the next one
    without continues persistently."""
    m = meshgen.jittered_square(40, periodic=True, seed=5)
    sch = vortex_scheme(dt=2e-3, reorder=1)
    a, b = Solver(m, sch, kernel_path=3), Solver(m, sch, kernel_path=2)
    b.set_launch_choices({"gradient": 2})
    b.set_persistent(True)
    for s in (a, b):
        s.initialize_solution(1, 0.0)
        s.time_integration(0.0, 3, vortex_error=True)
    assert np.array_equal(a.time_integration(0.0, 4), b.time_integration(0.0, 4))
    assert np.array_equal(a.cvar, b.cvar)
