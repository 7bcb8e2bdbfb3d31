"""LU in 32-column sub-panels with the rows in registers (subpanel.hip).

Tall m x n factorisations put every form of the panel and of its update at its
edges: one workgroup (256, 512 rows; 1024 in f32), 64 waves with one, two or four
rows per lane (4096, 8192, 16384), 128 waves (16384; 32768 in f32), one row more
than each, the form for still taller panels, a ragged last sub-panel (n not a
multiple of 32), sub-panels updated one by one (m <= 2048) and inside 128-column
panels with look-ahead (above).

Bars: the pivot vector equals the oracle's (lapack.rs:95-131), and with
k = min(m, n) and u the unit roundoff max |P A - L U| <= 8 k u max(|L| |U|), the
a-priori bound of Gaussian elimination (Higham, Accuracy and Stability, 9.3) with
room for the blocked order of the sums.
"""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (7, 5), (31, 33), (64, 64), (65, 96), (255, 40), (256, 40), (257, 64), (512, 70), (513, 40),
          (1024, 40), (1025, 40), (2048, 97), (2049, 200), (4096, 40), (4097, 150), (8192, 33), (8193, 140),
          (16384, 40), (16385, 33), (32768, 36), (32769, 33)]


@pytest.fixture(scope="module")
def L():
    from scirs_amd import linalg
    return linalg


def check(a, lu, perm):
    m, n = a.shape
    k = min(m, n)
    u = 2.0 ** (-53 if a.dtype == np.float64 else -24)
    low = np.tril(lu[:, :k].astype(np.float64), -1)
    low[np.arange(k), np.arange(k)] = 1.0
    up = np.triu(lu[:k].astype(np.float64))
    err = np.abs(a[perm].astype(np.float64) - low @ up).max()
    bound = 8 * k * u * (np.abs(low) @ np.abs(up)).max()
    assert err <= bound, (err, bound)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n", SHAPES)
def test_pivots_and_factors(L, m, n, dtype):
    a = np.random.default_rng(m + n).standard_normal((m, n)).astype(dtype)
    print(f"sub-panel LU {m} x {n} {dtype.__name__}", flush=True)
    lu, perm, _ = L.getrf(a)
    _, want, _ = oracle.lu_factor(a)
    assert np.array_equal(perm, want)
    check(a, lu, perm)


@pytest.mark.parametrize("m", [60, 500, 1500, 5000, 9000])
def test_first_of_equal_candidates(L, m):
    """Equal magnitudes: the first row wins (the strict '>' of lapack.rs:95-104),
    within a lane, a wave and across waves; values that differ in their last bits
    only (equal top words): the larger wins."""
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, 33))
    a[:, 0] = 0.5 * rng.choice([-1.0, 1.0], m)
    a[: m // 2, 0] = 0.25
    print(f"ties m={m}", flush=True)
    _, perm, _ = L.getrf(a)
    assert perm[0] == m // 2
    assert np.array_equal(perm, oracle.lu_factor(a)[1])
    a[:, 0] = (1.0 + rng.permutation(m) * 2.0 ** -50) * rng.choice([-1.0, 1.0], m)
    _, perm, _ = L.getrf(a)
    assert perm[0] == int(np.argmax(np.abs(a[:, 0])))
    assert np.array_equal(perm, oracle.lu_factor(a)[1])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,col", [(40, 0), (300, 39), (700, 33), (3000, 5), (9000, 37)])
def test_zero_column_stops(L, m, col, dtype):
    a = np.random.default_rng(m).standard_normal((m, 40)).astype(dtype)
    a[:, col] = 0.0
    print(f"zero column {col} of {m} {dtype.__name__}", flush=True)
    with pytest.raises(L.SingularError) as e:
        L.getrf(a)
    assert e.value.rc == col + 1
    lu, perm, _ = L.getrf(a[:, :col] if col else a[:, 1:])   # and the next call is whole again
    assert np.array_equal(perm, oracle.lu_factor(np.ascontiguousarray(a[:, :col] if col else a[:, 1:]))[1])


def test_large_pivot_divides_exactly(L):
    """Pivots whose reciprocal would be subnormal: the multipliers are still a / p."""
    a = np.random.default_rng(3).uniform(0.5, 1.0, (600, 1)) * 2.0 ** 1023
    lu, perm, _ = L.getrf(a)
    want, piv, _ = oracle.lu_factor(a)
    assert np.array_equal(perm, piv) and np.array_equal(lu, want)
