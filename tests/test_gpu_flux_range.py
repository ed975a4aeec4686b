"""The flux's own square roots and reciprocals over a wide range of magnitudes:
the Roe flux of states from 1e-100 to 1e100 against the oracle, whose operations
are the general ones.  Both round the same formula (some 150 operations, each off
by half an eps of a term within a few times the flux's scale: density, momentum or
enthalpy times velocity plus sound speed plus the entropy fix's width), which
bounds the difference by 1e-13 of that scale."""
import numpy as np
import pytest

from fvs2d_amd.solver import compute_flux_invscid
from oracle.oracle import roe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("decades", [1, 30, 100])
def test_flux_of_any_magnitude(decades):
    rng, n, g = np.random.default_rng(decades), 4000, 1.4
    rho, p = 10.0 ** rng.uniform(-decades, decades, (2, n))
    c = np.sqrt(g * p / rho)
    left = np.stack([rho, c * rng.uniform(-2, 2, n), c * rng.uniform(-2, 2, n), p], 1)
    right = left * (1.0 + rng.uniform(-0.5, 0.5, (n, 4)))
    right[::5, 1:3] = -left[::5, 1:3]
    right[::7] = left[::7]
    th = rng.uniform(0, 2 * np.pi, n)
    nxy = np.stack([np.cos(th), np.sin(th)], 1)
    f, ws = compute_flux_invscid(left, right, nxy[:, 0], nxy[:, 1], g)
    ref = [roe(g, left[i], right[i], *nxy[i]) for i in range(n)]
    c = 2.0 * np.maximum(c, np.sqrt(g * right[:, 3] / right[:, 0]))
    v = np.maximum(np.abs(left[:, 1:3]).sum(1), np.abs(right[:, 1:3]).sum(1))
    m = np.maximum(rho, right[:, 0]) * (v + c + 0.2)
    scale = np.stack([m, m * (v + c), m * (v + c), m * (2.5 * c * c + v * v)], 1)
    assert np.all(np.abs(f - np.array([r[0] for r in ref])) <= 1e-13 * scale)
    wr = np.array([r[1] for r in ref])
    assert np.all(np.abs(ws - wr) <= 1e-13 * (v + c))
