"""Persistent whole-step launches next to the other routes of a context: one that
changes between them and two kernels per stage continues from its current state,
bit for bit the kernels of kernel_path 3."""
import numpy as np
import pytest

from fvs2d_amd import _lib, meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu


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
