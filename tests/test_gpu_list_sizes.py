"""The whole-stage kernel's block lists do not grow with the widest stencil of the
mesh: the device memory of a context on a mesh with one node of many cells stays
within a quarter of the same mesh's without it."""
import gc

import pytest
import torch

from fvs2d_amd import meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme
from tests.test_gpu_large_nodes import hub_square

pytestmark = pytest.mark.gpu


def device_bytes(m, sch):
    gc.collect()  # contexts that earlier tests left behind
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    s = Solver(m, sch)
    used = free - torch.cuda.mem_get_info()[0]
    s.close()
    return used


@pytest.mark.parametrize("grad,limiter,k", [(3, 0, 50), (3, 1, 50), (2, 0, 30), (2, 1, 20)])
def test_one_large_node_costs_little_memory(grad, limiter, k):
    sch = vortex_scheme(dt=1e-3, reorder=1, grad_method=grad, limiter=limiter)
    device_bytes(meshgen.jittered_square(24, seed=1), sch)
    plain, hub = (device_bytes(m, sch) for m in (meshgen.jittered_square(256, seed=1), hub_square(256, k)))
    assert plain > 1 << 25 and hub < 1.25 * plain, (plain, hub)
