"""A rank-32 update adds its products to one another before they meet the element.

A leading identity block of 32 columns couples by entries 1/2 to a diagonal of 2^52
(f64; 2^23 in f32): each of the 32 products 1/4 vanishes when it is subtracted from the
diagonal by itself, their sum 8 does not.  Everything else stays below the last bit, so
the pivots are exactly 2^52 - 8 (and their roots, in the Cholesky factor)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BITS = {np.float64: 52, np.float32: 23}


def coupled(n, dtype):
    a = np.zeros((n, n), dtype)
    i = np.arange(n)
    a[i, i] = np.where(i < 32, 1.0, 2.0 ** BITS[dtype]).astype(dtype)
    a[32:, :32] = 0.5
    a[:32, 32:] = 0.5
    return a


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [160, 300, 1025, 2048])
def test_lu(n, dtype):
    from scirs_amd import linalg as L
    print(f"LU sums n={n} {dtype.__name__}", flush=True)
    lu, perm, _ = L.getrf(coupled(n, dtype))
    assert np.array_equal(perm, np.arange(n))
    assert (lu.diagonal()[32:] == dtype(2.0 ** BITS[dtype] - 8.0)).all()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [40, 64, 96, 128, 160, 700])
def test_cholesky(n, dtype):
    from scirs_amd import linalg as L
    print(f"Cholesky sums n={n} {dtype.__name__}", flush=True)
    low, _ = L.potrf(coupled(n, dtype))
    assert (low.diagonal()[32:] == np.sqrt(dtype(2.0 ** BITS[dtype] - 8.0))).all()
