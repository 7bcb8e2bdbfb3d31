"""LU panels with infinities and NaN, against the oracle (lapack.rs:95-143): a NaN compares
with nothing, so its row is not picked and spoils no other; a pivot row with an infinite
element spoils the rows below it, not the finished ones above.  And a column of zeros
reports a zero pivot."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu
CASES = [(m, dt) for m in (40, 300, 600, 1100, 3000, 9000) for dt in (np.float64, np.float32)] + [(20000, np.float32)]


@pytest.fixture(scope="module")
def L():
    from scirs_amd import linalg
    return linalg


def same(got, want, dtype):
    u = 2.0 ** (-53 if dtype == np.float64 else -24)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(want), want, 0))
    fin = np.isfinite(want)
    # the same eliminations in the same order, with and without fused products: 40 columns
    assert np.abs(got[fin] - want[fin]).max() <= 1e4 * u * np.abs(want[fin]).max()


@pytest.mark.parametrize("m,dtype", CASES)
@pytest.mark.parametrize("n", [8, 32, 39])
def test_nan_in_a_row_that_is_not_picked(L, m, n, dtype):
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n)).astype(dtype)
    a[m - 1, 3] = np.nan
    if m > 2 * n:
        a[m - 40, 5] = -np.nan
        a[m // 2, :] = np.nan
    print(f"NaN rows {m} x {n} {dtype.__name__}", flush=True)
    want, perm, _ = oracle.lu_factor(a)
    lu, p, _ = L.getrf(a)
    assert np.array_equal(p, perm)
    same(lu, want, dtype)


@pytest.mark.parametrize("m,dtype", CASES)
@pytest.mark.parametrize("n", [8, 32])
def test_infinite_element_of_a_pivot_row(L, m, n, dtype):
    rng = np.random.default_rng(m + n)
    a = rng.uniform(0.1, 1.0, (m, n)).astype(dtype)
    rows = rng.permutation(m)[:n]           # column j picks rows[j]
    a[rows, np.arange(n)] = 1000.0
    a[rows[n - 2], n - 1] = np.inf
    print(f"infinite element {m} x {n} {dtype.__name__}", flush=True)
    with np.errstate(all="ignore"):
        want, perm, _ = oracle.lu_factor(a)
    assert np.isfinite(want[: n - 2]).all() and np.array_equal(perm[: n - 1], rows[: n - 1])
    lu, p, _ = L.getrf(a)
    assert np.array_equal(p, perm)
    same(lu, want, dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [65, 513, 1025])
def test_zero_pivot_is_reported(L, m, dtype):
    a = np.zeros((m, 4), dtype)
    a[m - 1, 0] = 2.0                       # the only row of the last wave
    a[m - 1, 2] = 1.0 + 2.0 ** (-40 if dtype == np.float64 else -20)
    a[0, 1] = 1.0
    print(f"zero pivot of {m} {dtype.__name__}", flush=True)
    with pytest.raises(L.SingularError) as e:
        L.getrf(a)
    assert e.value.rc == 3 and e.value.info.pivot_value == 0.0


def test_square_with_a_nan_still_returns(L):
    """Every entry point ends, with a status or a result."""
    for n in (60, 700, 2500):
        a = np.random.default_rng(n).standard_normal((n, n))
        a[n // 3, n // 2] = np.nan
        b = np.ones(n)
        for name, f in (("gesv", L.gesv), ("gesv_ir", L.gesv_ir), ("getrf", lambda x, _: L.getrf(x))):
            print(f"{name} with a NaN n={n}", flush=True)
            try:
                f(a, b)
            except L.GpuSolveError as e:
                assert e.rc > 0
