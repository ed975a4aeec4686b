"""The whole-stage kernel (the default with LSQ gradients) against the
cell-by-cell gather and fused flux kernels (kernel_path 3), bit for bit: the
same arithmetic in the same order, so any difference is a wrong list entry or a
wrong index.  The cases are the edges of its blocks: cell counts around 64, 128
and 256, ranges cut to fit, every device order, halos read past the staged ones,
periodic meshes so small that a block wraps around itself, quadrilaterals, both
block shapes, and each limiter, weight exponent and integrator it is compiled
for.  The trajectory tests hold the arrangements to the oracle."""
import dataclasses

import numpy as np
import pytest

from fvs2d_amd import _lib, cases, meshgen
from fvs2d_amd.solver import BatchSolver, Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu

WHOLE = 8  # launch choice of the fused kernel: the whole stage in one kernel


def is_whole(s):
    try:
        s.set_launch_choices({"fused": WHOLE})
    except _lib.FvsError:
        return False
    return True


def both(m, sch, steps, expect=True, start=None, freeze=None):
    out = []
    for path in (0, 3):
        s = Solver(m, sch, kernel_path=path)
        if path == 0:
            assert is_whole(s) == expect
        if start is None:
            s.initialize_solution(1, 0.0)
        else:
            s.cvar = start
        n = s.time_integration(0.0, steps)
        if freeze:
            s.freeze_limiter(True)
            n = np.concatenate([n, s.time_integration(0.0, freeze)])
        out.append((s.cvar, n))
        s.close()
    assert np.all(np.isfinite(out[0][0]))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("reorder", [0, 1, 2])
@pytest.mark.parametrize("n", [3, 4, 5, 8, 9, 11, 12, 23, 40])
def test_block_edges(n, reorder):
    both(meshgen.jittered_square(n, periodic=True, seed=n), vortex_scheme(dt=0.005, reorder=reorder), 6)


@pytest.mark.parametrize("limiter", [0, 1, 2, 3])
@pytest.mark.parametrize("p", [0.0, 1.0, 2.0, 1.5])
@pytest.mark.parametrize("nn", [1, 0], ids=["nn", "fn"])
def test_limiters_and_weights(limiter, p, nn):
    """Unlimited with each weight, and each limiter (Van Albada on a uniform
    flow: its values leave [0, 1] elsewhere)."""
    m = meshgen.jittered_square(21, periodic=False, seed=2)
    kw = dict(vortex_K=0.0) if limiter == 3 else {}
    both(m, vortex_scheme(dt=0.003, reorder=1, lsq_p=p, lsq_nn=nn, limiter=limiter, **kw), 6)


@pytest.mark.parametrize("rk", [_lib.RK_CLASSIC, _lib.RK_SSP42, _lib.RK_SSP3, _lib.RK_SSP42_SO])
@pytest.mark.parametrize("steady", [0, 1])
def test_integrators(rk, steady):
    """Unsteady on the Dirichlet vortex (a global step is unstable in the
    O-grid's smallest cells), steady with local time steps on an O-grid."""
    if steady:
        m, sch = cases.naca(48, 25, cfl=0.3)
    else:
        m, sch = meshgen.jittered_square(26, periodic=False, seed=5), vortex_scheme(limiter=1, dt=1e-3, reorder=2)
    both(m, dataclasses.replace(sch, rk_scheme=rk, rk_order=4), 7, freeze=4)


def test_far_halo_cells():
    """Quads in a random order: every 64-cell block's halo exceeds what it
    stages, and the rest is read from memory."""
    m = meshgen.jittered_square(40, periodic=True, seed=1)
    quads = np.random.default_rng(3).permutation(m.ntri // 2)
    tri = m.cell_nodes.reshape(-1, 2, 3)[quads].reshape(-1)
    both(dataclasses.replace(m, cell_nodes=np.ascontiguousarray(tri)), vortex_scheme(dt=0.004, reorder=0), 5)


def test_random_cells_fall_back():
    m = meshgen.jittered_square(40, periodic=True, seed=1)
    order = np.random.default_rng(3).permutation(m.ntri)
    tri = m.cell_nodes.reshape(-1, 3)[order].reshape(-1)
    both(dataclasses.replace(m, cell_nodes=np.ascontiguousarray(tri)), vortex_scheme(dt=0.004, reorder=0), 5,
         expect=False)


@pytest.mark.parametrize("n", [9, 30])
def test_quadrilaterals(n):
    """A sheared grid of quadrilaterals with a Dirichlet outline whose corner
    cells are triangles, so that no cell has two boundary edges."""
    i, j = (a.ravel() for a in np.meshgrid(np.arange(n + 1), np.arange(n + 1)))
    xy = np.stack([-5 + 10 * i / n + 0.3 * j / n, -5 + 10 * j / n], 1).astype(float)
    qi, qj = (a.ravel() for a in np.meshgrid(np.arange(n), np.arange(n)))
    bl = qj * (n + 1) + qi
    br, tl, tr = bl + 1, bl + n + 1, bl + n + 2
    corner = (np.isin(qi, (0, n - 1)) & np.isin(qj, (0, n - 1)))
    main = corner & ((qi == 0) == (qj == 0))  # split bottom-left to top-right
    anti = corner & ~main
    tri = np.concatenate([np.stack([bl, br, tr], 1)[main], np.stack([bl, tr, tl], 1)[main],
                          np.stack([bl, br, tl], 1)[anti], np.stack([br, tr, tl], 1)[anti]])
    quad = np.stack([bl, br, tr, tl], 1)[~corner]
    side = np.stack([i == 0, i == n, j == 0, j == n], 1)
    edge = [(side[c] & np.roll(side[c], -1, axis=1)).any(axis=(1, 2)) for c in (tri, quad)]
    bnd = np.nonzero(np.concatenate(edge))[0].astype(np.int32)
    m = meshgen.Mesh(xy, len(tri), len(quad), np.concatenate([tri.ravel(), quad.ravel()]).astype(np.int32),
                     [("dirichlet", bnd)])
    for limiter in (0, 1):
        both(m, vortex_scheme(dt=0.01, reorder=1, limiter=limiter), 6)


def test_large_blocks():
    """65,536 cells of an O-grid, many of whose 128-cell ranges do not fit: the
    256-cell shape, with the limiter and after freezing it."""
    m, sch = cases.naca(256, 128)
    both(m, sch, 6, freeze=4)


def test_large_batch_masks():
    """The 256-cell shape in a batch: masked instances keep their state, the
    others are those of the unmasked batch."""
    conds = [((256, 128), (0.7, 1.0)), ((96, 50), (0.6, -1.0)), ((192, 97), (0.75, 2.0))]
    meshes = [cases.naca(n, l)[0] for (n, l), _ in conds]
    out = []
    for path in (0, 3):
        b = BatchSolver(meshes, [c for _, c in conds], cases.naca(32, 16, kernel_path=path)[1])
        b.initialize_freestream()
        b.batch_time_integration(0.0, 4)
        b.set_active([1, 0, 1])
        b.freeze_limiter_batch([0, 0, 1])
        b.batch_time_integration(0.0, 4)
        b.set_active([1, 1, 1])
        n = b.batch_time_integration(0.0, 3)
        out.append((b.cvar, n))
        b.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_launch_choices_switch():
    """Leaving the whole-stage kernel for two kernels per stage and coming back
    changes nothing but the launches; a choice that contradicts itself fails."""
    m = meshgen.jittered_square(70, periodic=True, seed=4)
    sch = vortex_scheme(dt=0.003, reorder=1)
    a, b = Solver(m, sch), Solver(m, sch)
    for s in (a, b):
        s.initialize_solution(1, 0.0)
    a.time_integration(0.0, 9)
    for ch in ({"gradient": 2}, {"fused": WHOLE}, {"gradient": 6, "fused": 4}):
        b.set_launch_choices(ch)
        b.time_integration(0.0, 3)
    assert np.array_equal(a.cvar, b.cvar)
    with pytest.raises(_lib.FvsError):
        b.set_launch_choices({"gradient": 2, "fused": WHOLE})
