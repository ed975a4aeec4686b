"""Residual norms of the time loop (src/runge_kutta.f90:169-184): each step's
squared increments leave the last stage as one sum per 64-cell slice, and the
pending steps are reduced together, so the cases here are the edges of that
arrangement: calls longer than the pending rows, cell counts that are no
multiple of 64, and batch instances whose boundaries fall inside slices
(several instances in one slice included).

The norms are compared with numpy's from the states before and after a step.
A relative difference of n eps from the order of the sum and a few eps from the
square root and division bound the disagreement: 2e-12 covers the 4,608 cells
of the largest mesh here."""
import numpy as np
import pytest

from fvs2d_amd import cases, meshgen
from fvs2d_amd.solver import BatchSolver, Solver
from tests.common import vortex_scheme

pytestmark = pytest.mark.gpu

TOL = 2e-12


def norms_of(u1, u0):
    return np.sqrt(np.mean((u1 - u0) ** 2, axis=0))


@pytest.mark.parametrize("kernel_path", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [5, 8, 21, 48])
def test_norms_match_states(n, kernel_path):
    m = meshgen.jittered_square(n, periodic=True, seed=n)
    s = Solver(m, vortex_scheme(dt=0.01), reorder=1, kernel_path=kernel_path)
    s.initialize_solution(1, 0.0)
    for _ in range(3):
        u0 = s.cvar
        got = s.time_integration(0.0, 1)[0]
        ref = norms_of(s.cvar, u0)
        assert np.all(np.abs(got - ref) <= TOL * ref)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("steps", [31, 33, 70])
def test_norm_rows_wrap(steps, graph):
    """One call of more steps than rows are pending gives the norms of that
    many calls of one step, bit for bit."""
    m, sch = cases.naca(24, 12, cfl=1.0)
    a, b = Solver(m, sch), Solver(m, sch)
    a.set_graph(graph)
    for s in (a, b):
        s.initialize_solution(1, 0.0)
    one = a.time_integration(0.0, steps)
    many = np.concatenate([b.time_integration(0.0, 1) for _ in range(steps)])
    assert np.array_equal(one, many) and np.array_equal(a.cvar, b.cvar)


@pytest.mark.parametrize("kernel_path", [0, 2])
@pytest.mark.parametrize("sizes", [[(8, 2), (8, 3), (10, 5), (24, 12)], [(32, 16), (48, 24)], [(9, 3)]],
                         ids=["several-per-slice", "aligned", "one-partial-slice"])
def test_instance_norms(sizes, kernel_path):
    meshes = [cases.naca(n, l)[0] for n, l in sizes]
    b = BatchSolver(meshes, [(0.5 + 0.05 * k, 1.0) for k in range(len(sizes))],
                    cases.naca(16, 8, cfl=0.5, limiter=0, kernel_path=kernel_path)[1])
    b.initialize_freestream()
    b.batch_time_integration(0.0, 2)
    o = b.cell_offsets
    u0 = b.cvar
    got = b.batch_time_integration(0.0, 1)[0]
    u1 = b.cvar
    for k in range(len(sizes)):
        ref = norms_of(u1[o[k]:o[k + 1]], u0[o[k]:o[k + 1]])
        assert np.all(np.abs(got[k] - ref) <= TOL * ref), k
    if len(sizes) > 1:
        # masked out, an instance repeats the norms of its last step
        b.set_active([0] + [1] * (len(sizes) - 1))
        n2 = b.batch_time_integration(0.0, 40)
        assert np.array_equal(n2[:, 0], np.tile(got[0], (40, 1)))
        assert not np.array_equal(n2[-1, 1], got[1])
