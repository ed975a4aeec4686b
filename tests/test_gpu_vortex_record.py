"""The vortex-error records of a run, reduced up to 32 steps at a time, against
those of the same steps taken one call at a time (whose times round differently:
1e-13), the single call of the last step, and the relations between the norms
(float64 sums: 1e-12)."""
import numpy as np
import pytest

from fvs2d_amd import meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu


# interior cells: fewer than one block of 256, one to eight blocks, more
@pytest.mark.parametrize("n,steps", [(6, 3), (13, 33), (30, 70), (100, 5)])
def test_records(n, steps):
    m = meshgen.jittered_square(n, periodic=False, seed=n)
    sch = vortex_scheme(dt=0.02 / n, reorder=1)
    a, b = Solver(m, sch), Solver(m, sch)
    for s in (a, b):
        s.initialize_solution(1, 0.0)
    _, rec = a.time_integration(0.0, steps, vortex_error=True)
    one = [b.time_integration(k * sch.dt, 1, vortex_error=True)[1][0] for k in range(steps)]
    assert np.array_equal(a.cvar, b.cvar)
    t_end = (steps - 1) * sch.dt + sch.dt
    assert np.array_equal(rec[-1], np.asarray(a.error_isentropic_vortex(t_end)).ravel())
    assert np.allclose(rec, np.array(one), rtol=1e-13, atol=0.0)
    e = rec[-1][:12].reshape(4, 3)
    assert np.all(e[:, 0] >= e[:, 2]) and np.all(e[:, 2] >= e[:, 1] * (1 - 1e-12))  # max >= rms >= mean
    assert np.isclose(rec[-1][12] ** 2, (e[:, 2] ** 2).sum(), rtol=1e-12, atol=0.0)
