"""The chained FP64 triangular solve divides by a reciprocal taken ahead and
corrected, and by true division where a block's diagonal leaves the range in
which that reciprocal is a normal number."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 129])
@pytest.mark.parametrize("nrhs", [1, 2])
@pytest.mark.parametrize("lower", [True, False])
def test_rows_scaled_past_the_reciprocals_range(n, nrhs, lower):
    """Rows scaled by 2^980: every operation scales exactly, so the solution
    is that of the unscaled triangle, within the bar of the solver's other
    tests (1e-12 max|x| on a well-conditioned triangle)."""
    from scirs_amd import linalg as L
    rng = np.random.default_rng(n + nrhs)
    a = rng.standard_normal((n, n)) / np.sqrt(n)
    a = np.tril(a) if lower else np.triu(a)
    np.fill_diagonal(a, 1.0 + rng.random(n))
    b = rng.standard_normal((n, nrhs))
    xo = np.stack([oracle.solve_triangular(a, np.ascontiguousarray(b[:, j]), lower, False) for j in range(nrhs)], 1)
    x0, _ = L.trsv(a, b, lower, False)
    rows = [0, n // 2, n - 1]
    a[rows] *= 2.0 ** 980
    b[rows] *= 2.0 ** 980
    x1, _ = L.trsv(a, b, lower, False)
    for x in (x0, x1):
        assert (np.abs(x - xo).max(axis=0) <= 1e-12 * np.abs(xo).max(axis=0)).all()


def test_infinite_and_overflowing_entries():
    """An entry that overflows is infinite, as in the division, and leaves the
    entries before it alone."""
    from scirs_amd import linalg as L
    n = 100
    a = np.eye(n)
    a[70, 70] = 1e-9
    b = np.ones(n)
    b[70] = 1e305
    x, _ = L.trsv(a, b, True, False)
    assert np.array_equal(x.ravel(), oracle.solve_triangular(a, b, True, False), equal_nan=True)
    assert (x.ravel()[:70] == 1.0).all() and np.isposinf(x.ravel()[70])
