"""The QR panel at the edges of its workgroups (256 rows each, eight sums per thread and
pass) and of its 32-column width, through least squares.

Bar: both solvers are backward stable, so |x - x_lapack| <= 8 m 2^-53 kappa_2(A)
max|x_lapack| for the small residuals here (Gaussian A, kappa below 10)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(32, 1), (256, 32), (257, 33), (300, 31), (2048, 36), (2049, 64), (8193, 35),
                                   (16384, 34)])
def test_panel_edges(shape):
    from scirs_amd import linalg as L
    m, n = shape
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n))
    a[n // 2] += 1.0
    b = a @ rng.standard_normal(n) + 0.1 * rng.standard_normal(m)
    print(f"lstsq {m} x {n}", flush=True)
    x = np.asarray(L.lstsq(a, b)[0]).ravel()
    xr = np.linalg.lstsq(a, b, rcond=None)[0]
    bar = 8 * m * 2.0 ** -53 * np.linalg.cond(a)
    assert np.abs(x - xr).max() <= bar * np.abs(xr).max()
