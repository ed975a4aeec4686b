"""The whole-stage kernel with Green-Gauss gradients (cell-based 1, node-based 2)
against the gradient and fused flux kernels (kernel_path 3), bit for bit: the same
functions in the same order, so any difference is a wrong list entry or index.
Cases: the edges of its blocks, every device order, meshes so small that a block
wraps around itself, quadrilaterals, nodes of many cells, both block shapes, each
limiter and integrator, frozen limiters, and the residual call."""
import dataclasses

import numpy as np
import pytest

from fvs2d_amd import _lib, cases, meshgen
from fvs2d_amd.solver import Solver
from tests.common import vortex_scheme
from tests.test_gpu_whole_stage import WHOLE, both, is_whole

pytestmark = pytest.mark.gpu
GM = pytest.mark.parametrize("gm", [1, 2], ids=["ggcb", "ggnb"])


@GM
@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("n,reorder", [(3, 1), (4, 0), (5, 2), (8, 1), (9, 0), (12, 2), (23, 1), (41, 0), (150, 1)])
def test_block_edges(gm, limiter, n, reorder):
    """In the mesh's own order the blocks are strips, whose second ring fits LDS
    only up to a width: wider meshes keep the two kernels."""
    both(meshgen.jittered_square(n, periodic=True, seed=n),
         vortex_scheme(dt=0.04 / n, reorder=reorder, grad_method=gm, limiter=limiter), 5,
         expect=(n, reorder) != (41, 0) or (gm == 1 and limiter == 0))


@GM
@pytest.mark.parametrize("limiter", [0, 1, 2, 3])
def test_limiters(gm, limiter):
    m = meshgen.jittered_square(21, periodic=False, seed=2)
    kw = dict(vortex_K=0.0) if limiter == 3 else {}
    both(m, vortex_scheme(dt=0.003, reorder=1, grad_method=gm, limiter=limiter, **kw), 6, freeze=3 if limiter else None)


@GM
@pytest.mark.parametrize("rk", [_lib.RK_CLASSIC, _lib.RK_SSP42, _lib.RK_SSP42_SO])
@pytest.mark.parametrize("steady", [0, 1])
def test_integrators(gm, rk, steady):
    if steady:
        m, sch = cases.naca(48, 25, cfl=0.3)
    else:
        m, sch = meshgen.jittered_square(26, periodic=False, seed=5), vortex_scheme(limiter=1, dt=1e-3, reorder=2)
    both(m, dataclasses.replace(sch, grad_method=gm, rk_scheme=rk, rk_order=4), 7, freeze=4)


@GM
@pytest.mark.parametrize("limiter", [0, 1])
def test_large_blocks(gm, limiter):
    """65,536 cells of an O-grid: ranges of 128 cells that do not fit."""
    m, sch = cases.naca(256, 128, cfl=0.3)
    both(m, dataclasses.replace(sch, grad_method=gm, limiter=limiter), 4)


@GM
@pytest.mark.parametrize("limiter", [0, 1])
def test_quadrilaterals(gm, limiter):
    """Quadrilaterals with a Dirichlet outline whose corner cells are triangles, so
    that no cell has two boundary edges."""
    n = 30
    i, j = (a.ravel() for a in np.meshgrid(np.arange(n + 1), np.arange(n + 1)))
    xy = np.stack([-5 + 10 * i / n + 0.3 * j / n, -5 + 10 * j / n], 1).astype(float)
    qi, qj = (a.ravel() for a in np.meshgrid(np.arange(n), np.arange(n)))
    bl = qj * (n + 1) + qi
    br, tl, tr = bl + 1, bl + n + 1, bl + n + 2
    corner = (np.isin(qi, (0, n - 1)) & np.isin(qj, (0, n - 1)))
    main = corner & ((qi == 0) == (qj == 0))
    anti = corner & ~main
    tri = np.concatenate([np.stack([bl, br, tr], 1)[main], np.stack([bl, tr, tl], 1)[main],
                          np.stack([bl, br, tl], 1)[anti], np.stack([br, tr, tl], 1)[anti]])
    quad = np.stack([bl, br, tr, tl], 1)[~corner]
    side = np.stack([i == 0, i == n, j == 0, j == n], 1)
    edge = [(side[c] & np.roll(side[c], -1, axis=1)).any(axis=(1, 2)) for c in (tri, quad)]
    bnd = np.nonzero(np.concatenate(edge))[0].astype(np.int32)
    m = meshgen.Mesh(xy, len(tri), len(quad), np.concatenate([tri.ravel(), quad.ravel()]).astype(np.int32),
                     [("dirichlet", bnd)])
    both(m, vortex_scheme(dt=0.01, reorder=1, grad_method=gm, limiter=limiter), 6)


@GM
def test_random_cells_fall_back(gm):
    m = meshgen.jittered_square(40, periodic=True, seed=1)
    order = np.random.default_rng(3).permutation(m.ntri)
    tri = m.cell_nodes.reshape(-1, 3)[order].reshape(-1)
    both(dataclasses.replace(m, cell_nodes=np.ascontiguousarray(tri)),
         vortex_scheme(dt=0.004, reorder=0, grad_method=gm), 5, expect=False)


@GM
@pytest.mark.parametrize("limiter", [0, 1])
def test_residual_and_choices(gm, limiter):
    """The residual, wave speeds, gradient and limiter of both forms; leaving the
    whole-stage kernel and coming back changes nothing."""
    m = meshgen.jittered_square(37, periodic=True, seed=4)
    sch = vortex_scheme(dt=0.003, reorder=1, grad_method=gm, limiter=limiter)
    a, b = Solver(m, sch), Solver(m, sch, kernel_path=3)
    for s in (a, b):
        s.initialize_solution(1, 0.0)
    assert is_whole(a)
    for x, y in zip(a.compute_residual(0.0), b.compute_residual(0.0)):
        assert np.array_equal(x, y)
    b.time_integration(0.0, 6)
    for ch in ({"gradient": 2 if limiter else 0}, {"fused": WHOLE}, {"fused": 1}):
        a.set_launch_choices(ch)
        a.time_integration(0.0, 2)
    assert np.array_equal(a.cvar, b.cvar)
    assert np.array_equal(a.compute_gradient_cellcntr(), b.compute_gradient_cellcntr())
    a.close()
    b.close()
