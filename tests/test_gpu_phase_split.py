"""The phase timers of whole-stage launches are measured on the device: what a
limiter adds is gradient time, so its phase takes a larger part of the same
mesh's launches with it than without (by 10% and more: the limiter is some 150
operations on each of the cells with a gradient)."""
import numpy as np
import pytest

from fvs2d_amd import meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grad", [1, 2, 3])
def test_limiter_shows_in_the_gradient_phase(grad):
    m = meshgen.jittered_square(200, periodic=True, seed=1)
    part = []
    for limiter in (0, 1):
        s = Solver(m, vortex_scheme(dt=1e-3, reorder=1, limiter=limiter, grad_method=grad))
        s.initialize_solution(1, 0.0)
        s.time_integration(0.0, 20)
        s.set_phase_timers(True)
        s.time_integration(0.0, 40)
        t = s.phase_times()
        assert np.all(np.isfinite(t)) and t[0] > 0 and t[2] > 0 and t[1] == 0
        part.append(t[0] / (t[0] + t[2]))
    assert part[1] > 1.1 * part[0]
