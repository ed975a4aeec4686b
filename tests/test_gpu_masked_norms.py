"""A masked batch instance repeats the residual norms of its last step whether
or not the call that took that step asked for them: calls with whole-mesh norms
or with none at all, as single launches, captured graphs and persistent
launches, with instances that share 64-cell slices.  Bit for bit the norms of a
batch that asks every time."""
import numpy as np
import pytest

from fvs2d_amd import cases
from fvs2d_amd._lib import check
from fvs2d_amd.solver import BatchSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("launch", ["plain", "graph", "persistent"])
@pytest.mark.parametrize("call", ["mesh", "none"])
def test_masked_instance_keeps_norms_nobody_asked_for(call, launch):
    meshes = [cases.naca(n, l)[0] for n, l in [(8, 2), (8, 3), (10, 5), (24, 12)]]
    sch = cases.naca(16, 8, cfl=0.02, limiter=0, kernel_path=2 if launch == "persistent" else 0)[1]
    a, b = (BatchSolver(meshes, [(0.5 + 0.05 * k, 1.0) for k in range(4)], sch) for _ in range(2))
    for s in (a, b):
        if launch == "graph":
            s.set_graph(True)
        if launch == "persistent":
            s.set_persistent(True)
        s.initialize_freestream()
    if call == "mesh":
        a.time_integration(0.0, 41)
    else:
        check(a._L.fvs_batch_time_integration(a._h, 0.0, 41, None))
    last = b.batch_time_integration(0.0, 41)[-1]
    for s in (a, b):
        s.set_active([0, 1, 0, 1])
    got, ref = a.batch_time_integration(0.0, 40), b.batch_time_integration(0.0, 40)
    assert np.all(last > 0.0)
    for k in (0, 2):
        assert np.array_equal(got[:, k], np.tile(last[k], (40, 1)))
    assert np.array_equal(got, ref)
