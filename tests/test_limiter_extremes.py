"""The limiter value of a cell from the largest rise and the largest fall of a
variable over its faces, as the kernels form it, against every face's candidate:
both limiter forms, over increments and bounds of any size, zeros included.  The
two differ at most where candidates are within rounding of each other: 4 ulp."""
import numpy as np
import pytest


def venkat(a, b, eps2):
    return ((a * a + eps2) + 2.0 * b * a) / (a * a + 2.0 * (b * b) + a * b + eps2)


@pytest.mark.parametrize("form", ["venkat", "barth"])
@pytest.mark.parametrize("faces", [1, 3, 4])
def test_extreme_faces_suffice(form, faces):
    rng = np.random.default_rng(faces)
    n = 200000
    size = 10.0 ** rng.uniform(-12, 3, (faces, n))
    b = size * rng.choice([-1.0, 0.0, 1.0], (faces, n), p=[0.45, 0.1, 0.45])
    dmax = 10.0 ** rng.uniform(-12, 3, n) * rng.choice([0.0, 1.0], n, p=[0.1, 0.9])
    dmin = -(10.0 ** rng.uniform(-12, 3, n)) * rng.choice([0.0, 1.0], n, p=[0.1, 0.9])
    eps2 = 10.0 ** rng.uniform(-12, 0, n)

    def value(b):
        a = np.where(b > 0, dmax, dmin)
        with np.errstate(all="ignore"):
            l = venkat(a, b, eps2) if form == "venkat" else a / b
        return np.where(b == 0, 1.0, np.minimum(1.0, l))

    every = np.min([value(x) for x in b], axis=0)
    few = np.minimum(value(np.maximum(0.0, b.max(0))), value(np.minimum(0.0, b.min(0))))
    assert np.all(np.abs(every - few) <= 4 * np.finfo(float).eps * np.maximum(every, few))
