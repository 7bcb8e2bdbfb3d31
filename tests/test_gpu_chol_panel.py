"""The Cholesky panel kernel (potrf.hip, chol_panel_kernel) and the small-tile update
(gemm_mfma.hip, gemm_nt64_kernel) at their edges: orders around the 32-column steps,
the 128-column panels and 64- and 128-row tiles, ragged last panels, the order where
the update changes from small to large tiles, f64 and f32, and a diagonal that turns
negative in each 32-column step and row group.

Bars: with u the unit roundoff, max |A - L L^T| <= 4 n u max(diag A), the a-priori
bound of Cholesky (Higham, Accuracy and Stability, 10.1); the strict upper triangle of
L is zero; the failing row equals the oracle's (lapack.rs:661-670).
"""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    from scirs_amd import linalg
    return linalg


def definite(n, dtype):
    g = np.random.default_rng(n).standard_normal((n, n))
    return (g @ g.T / n + np.eye(n)).astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 63, 65, 96, 97, 127, 128, 129, 160, 161, 255, 257, 385, 1023, 2049,
                               2177])
def test_factor(L, n, dtype):
    a = definite(n, dtype)
    print(f"cholesky panel n={n} {dtype.__name__}", flush=True)
    low, _ = L.potrf(a)
    assert not np.triu(low, 1).any()
    low = low.astype(np.float64)
    u = 2.0 ** (-53 if dtype == np.float64 else -24)
    err = np.abs(np.tril(a.astype(np.float64) - low @ low.T)).max()
    assert err <= 4 * n * u * a.diagonal().max(), err


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,row", [(1, 0), (40, 0), (40, 39), (128, 31), (128, 32), (128, 100), (200, 127), (200, 128),
                                   (300, 299), (700, 160), (700, 255)])
def test_first_row_that_fails(L, n, row, dtype):
    a = definite(n, dtype)
    a[row, row] = -0.5
    print(f"cholesky failing row {row} of {n} {dtype.__name__}", flush=True)
    with pytest.raises(L.NotPositiveDefiniteError) as e:
        L.potrf(a)
    with pytest.raises(oracle.OracleError) as o:
        oracle.cholesky(a)
    assert e.value.rc == o.value.code == row + 1
    L.potrf(definite(n, dtype))   # and the next call is whole again
