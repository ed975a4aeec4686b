"""Per-cell arrays in and out of the context in the caller's order, and the
residual evaluation by the whole-stage kernel.  The residual is compared bit for
bit with the cell-by-cell gather and fused flux kernels (kernel_path 3): the same
arithmetic in the same order.  A state written and read back is the same bits,
and a renumbered mesh (reorder 1, 2) gives every cell's values at the cell's own
index: those of reorder 0 up to the rounding of another edge orientation, which
a flux or a gradient of at most four edges turns into no more than a few units
in the last place of the largest term; 1e-11 of the field's largest value holds
two orders of margin over that (the limiter's ratios are compared with 1e-9)."""
import numpy as np
import pytest

from fvs2d_amd import cases, meshgen
from fvs2d_amd.solver import BatchSolver, Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu


def rough_state(s, seed=0):
    """The vortex with a few percent of noise in every cell."""
    s.initialize_solution(1, 0.0)
    u = s.cvar
    u *= 1.0 + 0.02 * np.random.default_rng(seed).standard_normal(u.shape)
    s.cvar = u
    return u


@pytest.mark.parametrize("limiter", [0, 1])
@pytest.mark.parametrize("reorder", [0, 1, 2])
@pytest.mark.parametrize("n,periodic", [(3, True), (5, True), (8, False), (9, False), (11, True), (23, False)])
def test_residual(n, periodic, reorder, limiter):
    m = meshgen.jittered_square(n, periodic=periodic, seed=n)
    out = []
    for path in (0, 2, 3):
        s = Solver(m, vortex_scheme(reorder=reorder, limiter=limiter, kernel_path=path))
        u = rough_state(s)
        r = s.compute_residual(0.25)
        dt = s.compute_local_time()
        assert np.array_equal(s.cvar, u)
        s.time_integration(0.25, 2)
        s.freeze_limiter(True)
        out.append((*r, dt, s.cvar, *s.compute_residual(0.5)))
        s.close()
    for a, b, c in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, c) and np.array_equal(b, c)


def test_residual_steady_large_blocks_and_masks():
    """The 256-cell shape in a batch whose middle instance is stopped: every
    instance's residual, as without the mask."""
    meshes = [cases.naca(*d)[0] for d in ((256, 128), (96, 50), (192, 97))]
    conds = [(0.7, 1.0), (0.6, -1.0), (0.75, 2.0)]
    out = []
    for path in (0, 3):
        b = BatchSolver(meshes, conds, cases.naca(32, 16, kernel_path=path)[1])
        b.initialize_freestream()
        b.batch_time_integration(0.0, 3)
        r = b.compute_residual(0.0)
        if path == 0:
            b.set_active([1, 0, 1])
            assert all(np.array_equal(x, y) for x, y in zip(r, b.compute_residual(0.0)))
            b.set_active([1, 1, 1])
        out.append((*r, b.batch_time_integration(0.0, 2), b.cvar))
        b.close()
    assert all(np.array_equal(x, y) for x, y in zip(*out))


@pytest.mark.parametrize("grad", [1, 2, 3])
@pytest.mark.parametrize("n", [3, 9, 12, 40])
def test_caller_order(n, grad):
    m = meshgen.jittered_square(n, periodic=False, seed=n)
    ref = None
    for reorder in (0, 1, 2):
        s = Solver(m, vortex_scheme(reorder=reorder, limiter=1, grad_method=grad))
        u = rough_state(s, 3)
        assert np.array_equal(s.cvar, u)
        w = s.cvar2pvar()
        g = s.compute_gradient_cellcntr()
        g1 = s.gradient_cellcntr_1var(w[:, 3])
        got = (w, g, g1, *s.compute_residual(0.0), s.compute_gradient_limiter())
        s.close()
        ref = ref or got
        for k, (a, b) in enumerate(zip(got, ref)):
            assert np.abs(a - b).max() <= (1e-9 if k == 5 else 1e-11) * np.abs(b).max()
