"""Limiter values of a masked batch instance outlive everything that is asked of
the context meanwhile: the instance resumes with its limiter frozen at the
values of its last evaluation, bit for bit as if nothing had been asked.  The
instances share blocks, so the masked cells are part of the launches between."""
import numpy as np
import pytest

from fvs2d_amd import _lib, cases
from fvs2d_amd.solver import BatchSolver

pytestmark = pytest.mark.gpu

ASK = {
    "state": lambda s: s.cvar,
    "primitives": lambda s: s.cvar2pvar(),
    "gradient": lambda s: s.compute_gradient_cellcntr(),
    "scalar gradient": lambda s: s.gradient_cellcntr_1var(np.linspace(-1.0, 1.0, s.ncells)),
    "forces": lambda s: s.wall_forces_batch(),
    "limiter": lambda s: s.compute_gradient_limiter(),
    "residual": lambda s: s.compute_residual(0.0),
}
ROUTES = {"whole-stage": (0, None), "two-kernels": (0, {"gradient": 2}), "primitive": (2, None), "gather": (3, None)}


@pytest.mark.parametrize("route", list(ROUTES))
@pytest.mark.parametrize("rk", [_lib.RK_SSP3, _lib.RK_SSP42_SO, _lib.RK_SSP42])
@pytest.mark.parametrize("ask", list(ASK))
def test_queries_leave_frozen_limiters_alone(ask, rk, route):
    path, choices = ROUTES[route]
    meshes = [cases.naca(n, l)[0] for n, l in [(24, 12), (20, 11)]]
    out = []
    for query in (None, ASK[ask]):
        b = BatchSolver(meshes, [(0.7, 1.0), (0.6, -1.0)], cases.naca(16, 8, cfl=0.5, rk_scheme=rk, kernel_path=path)[1])
        if choices:
            b.set_launch_choices(choices)
        b.initialize_freestream()
        b.batch_time_integration(0.0, 20)
        b.set_active([0, 1])
        if query:
            query(b)
        b.batch_time_integration(0.0, 3)
        b.set_active([1, 1])
        b.freeze_limiter_batch([1, 0])
        n = b.batch_time_integration(0.0, 4)
        out.append((b.cvar, n))
        b.close()
    assert np.all(np.isfinite(out[0][0]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
