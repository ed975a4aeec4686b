"""Meshes with a node of many cells: the states are those of kernel_path 3 bit
for bit, and a node of more cells than any block holds leaves the mesh to two
kernels per stage."""
import numpy as np
import pytest

from fvs2d_amd import _lib, meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu


def hub_square(n, k):
    """The n x n square (Dirichlet outline) with its middle k x k quads replaced
    by the 4 k triangles around the middle node."""
    m = meshgen.jittered_square(n, periodic=False, seed=n)
    a, b = n // 2 - k // 2, n // 2 - k // 2 + k
    q = np.arange(m.ntri) // 2
    qi, qj = q % n, q // n
    keep = ~((qi >= a) & (qi < b) & (qj >= a) & (qj < b))
    tri = m.cell_nodes.reshape(-1, 3)
    ring = np.concatenate([[(a, i) for i in range(a, b)], [(j, b) for j in range(a, b)],
                           [(b, i) for i in range(b, a, -1)], [(j, a) for j in range(b, a, -1)]])
    ring = ring[:, 0] * (n + 1) + ring[:, 1]
    hub = (n // 2) * (n + 1) + n // 2
    fan = np.stack([np.full(4 * k, hub), ring, np.roll(ring, -1)], 1)
    cells = np.concatenate([tri[keep], fan])
    used, ids = np.unique(cells, return_inverse=True)
    renumber = np.cumsum(keep) - 1
    bnd = renumber[m.boundaries[0][1]].astype(np.int32)
    return meshgen.Mesh(m.xy[used], len(cells), 0, ids.reshape(-1).astype(np.int32), [("dirichlet", bnd)])


def disk(cells):
    """Triangles around one node."""
    t = 2 * np.pi * np.arange(cells) / cells
    xy = np.concatenate([[[0.0, 0.0]], 5 * np.stack([np.cos(t), np.sin(t)], 1)])
    i = np.arange(cells)
    tri = np.stack([0 * i, 1 + i, 1 + (i + 1) % cells], 1)
    return meshgen.Mesh(xy, cells, 0, tri.ravel().astype(np.int32), [("dirichlet", i.astype(np.int32))])


@pytest.mark.parametrize("reorder", [0, 1, 2])
@pytest.mark.parametrize("grad,limiter,k", [(3, 0, 12), (3, 1, 12), (3, 0, 50), (3, 1, 50), (1, 1, 12), (2, 0, 6),
                                            (2, 0, 12), (2, 1, 12), (2, 0, 30), (2, 1, 30)])
def test_states_around_a_large_node(grad, limiter, k, reorder):
    out = []
    for path in (0, 3):
        s = Solver(hub_square(60, k), vortex_scheme(dt=2e-4, reorder=reorder, grad_method=grad, limiter=limiter,
                                                    kernel_path=path))
        s.initialize_solution(1, 0.0)
        n = s.time_integration(0.0, 6)
        out.append((s.cvar, n))
    assert np.all(np.isfinite(out[0][0]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_node_of_more_cells_than_a_block():
    out = []
    for path in (0, 3):
        s = Solver(disk(9001), vortex_scheme(dt=1e-5, reorder=1, grad_method=2, kernel_path=path))
        if path == 0:
            with pytest.raises(_lib.FvsError, match="whole-stage"):
                s.set_launch_choices({"fused": 8})
        s.initialize_solution(1, 0.0)
        s.time_integration(0.0, 3)
        out.append(s.cvar)
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])
