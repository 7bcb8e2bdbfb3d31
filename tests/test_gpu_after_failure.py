"""A factorisation that fails leaves nothing behind: the calls after it are checked by
their results, after failures in the first and in later panels, with fewer and with more
panel workgroups than fit on the device at once (512; 32 rows each).

Bars: the normwise backward error of a solve <= 4 n 2^-53; max |A - L L^T| <= 4 n u
max(diag A) (Higham, Accuracy and Stability, 10.1); max |P A - L U| <= 8 n u max(|L| |U|)
(9.3)."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu
U64 = 2.0 ** -53


@pytest.fixture(scope="module")
def L():
    from scirs_amd import linalg
    return linalg


def solves_are_whole(L, n, nrhs=2):
    """LU and Cholesky solves on the device: the Cholesky panel's diagonal blocks and the
    LU update's first strip are what a wrong arrival count would spoil."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    m = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    spd = m @ m.T / n + torch.eye(n, dtype=torch.float64, device="cuda")
    b = torch.randn(n, nrhs, dtype=torch.float64, device="cuda", generator=g)
    x = torch.empty_like(b)
    for what, solve, a in (("posv", L.posv_dev, spd), ("gesv", L.gesv_dev, m), ("posv", L.posv_dev, spd)):
        solve(a, b, x)
        r = b - a @ x
        eta = float(r.abs().max() / (a.abs().sum(dim=1).max() * x.abs().max() + b.abs().max()))
        assert eta <= 4 * n * U64, (what, n, eta)


def factors_are_whole(L, n, dtype):
    rng = np.random.default_rng(n)
    g = rng.standard_normal((n, n))
    a = (g @ g.T / n + np.eye(n)).astype(dtype)
    u = 2.0 ** (-53 if dtype == np.float64 else -24)
    low, _ = L.potrf(a)
    assert not np.triu(low, 1).any()
    low = low.astype(np.float64)
    assert np.abs(np.tril(a.astype(np.float64) - low @ low.T)).max() <= 4 * n * u * a.diagonal().max()
    a = g.astype(dtype)
    lu, perm, _ = L.getrf(a)
    low, up = np.tril(lu.astype(np.float64), -1) + np.eye(n), np.triu(lu.astype(np.float64))
    assert np.abs(a[perm].astype(np.float64) - low @ up).max() <= 8 * n * u * (np.abs(low) @ np.abs(up)).max()
    assert np.array_equal(perm, oracle.lu_factor(a)[1])


@pytest.mark.parametrize("n,row", [(4096, 3), (4096, 2100), (17000, 0), (17000, 5), (17000, 8200)])
def test_cholesky_fails_on_the_device(L, n, row):
    import torch
    print(f"device Cholesky failing at row {row} of {n}", flush=True)
    a = torch.eye(n, dtype=torch.float64, device="cuda").mul_(2.0)
    a[row, row] = -1.0
    b = torch.ones(n, 1, dtype=torch.float64, device="cuda")
    x = torch.empty_like(b)
    for _ in range(3):
        with pytest.raises(L.NotPositiveDefiniteError) as e:
            L.posv_dev(a, b, x)
        assert e.value.rc == row + 1
    del a
    solves_are_whole(L, 1500)
    solves_are_whole(L, 4500, 1)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,row", [(40, 0), (200, 128), (700, 255)])
def test_cholesky_fails_on_the_host(L, n, row, dtype):
    a = (2.0 * np.eye(n)).astype(dtype)
    a[row, row] = -0.5
    print(f"host Cholesky failing at row {row} of {n} {dtype.__name__}", flush=True)
    with pytest.raises(L.NotPositiveDefiniteError) as e:
        L.potrf(a)
    assert e.value.rc == row + 1
    factors_are_whole(L, n, dtype)
    factors_are_whole(L, 300, dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,col", [(40, 0), (300, 39), (700, 33), (3000, 5), (9000, 37)])
def test_singular_column(L, m, col, dtype):
    a = np.random.default_rng(m).standard_normal((m, 40)).astype(dtype)
    a[:, col] = 0.0
    print(f"LU with zero column {col} of {m} {dtype.__name__}", flush=True)
    with pytest.raises(L.SingularError) as e:
        L.getrf(a)
    assert e.value.rc == col + 1
    factors_are_whole(L, 300, dtype)
    factors_are_whole(L, 1100, dtype)
