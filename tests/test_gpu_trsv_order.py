"""The chained triangular solve subtracts a block's products in the order of the columns.

The triangles here hold identity diagonal blocks and couplings of large entries of
alternating sign whose neighbours almost cancel.  In column order every partial sum is a
whole number that fits the significand, so the solution is exact; summed in any two halves
the partial sums outgrow it and round."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bits", [(np.float64, 52), (np.float32, 23)])
@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("nrhs", [1, 2, 3])
@pytest.mark.parametrize("n", [128, 100])
def test_neighbouring_columns_cancel(n, nrhs, lower, dtype, bits):
    from scirs_amd import linalg as L
    rng = np.random.default_rng(n + nrhs)
    print(f"substitution order n={n} nrhs={nrhs} lower={lower} {dtype.__name__}", flush=True)
    big = 2.0 ** (bits - 1)
    head, tail = slice(0, 64), slice(64, n)             # the solver's blocks of 64 rows
    rows, cols = (tail, head) if lower else (head, tail)
    m, k = len(range(n)[rows]), len(range(n)[cols])
    odd = rng.integers(1, 8, (m, k // 2)).astype(dtype)
    couple = np.empty((m, k), dtype)
    couple[:, 0::2] = big
    couple[:, 1::2] = odd - dtype(big)
    a = np.eye(n, dtype=dtype)
    a[rows, cols] = couple
    b = np.zeros((n, nrhs), dtype)
    b[cols] = 1 + np.arange(nrhs, dtype=dtype) % 2      # x there: 1, 2, 1, ...
    want = b.copy()
    want[rows] = -odd.sum(axis=1, dtype=dtype)[:, None] * b[cols][:1]
    x, _ = L.trsv(a, b, lower, False, dtype=dtype)
    assert np.array_equal(x, want)
