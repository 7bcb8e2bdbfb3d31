"""Batched solves at the edges of the 16-row blocks and 64-row register sets, and batches
in which some systems leave FP32.

Bar, as for the other batched solves: normwise backward error <= 8 n 2^-53 per right-hand
side (the refinement stops at n 2^-53; the factor covers the test's own residual)."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu
U64 = 2.0 ** -53


def system(rng, n, spd):
    g = rng.standard_normal((n, n))
    return 0.5 * (g @ g.T + (g @ g.T).T) / n + np.eye(n) if spd else g + 2.0 * np.diag(rng.choice([-1.0, 1.0], n))


def check(a, x, b):
    n = a.shape[0]
    r = b - a @ x
    den = np.abs(a).sum(axis=1).max() * np.abs(x).max(axis=0) + np.abs(b).max(axis=0)
    assert (np.abs(r).max(axis=0) <= 8 * n * U64 * den).all(), (n, (np.abs(r).max(axis=0) / den).max() / U64)


@pytest.mark.parametrize("nrhs", [1, 4, 5, 16])
@pytest.mark.parametrize("spd", [0, 1])
def test_block_and_register_set_edges(nrhs, spd):
    from scirs_amd import linalg as L
    sizes = [1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 80, 81, 127, 128, 129, 191, 192, 193, 240, 241, 255, 256]
    rng = np.random.default_rng(10 * nrhs + spd)
    As = [system(rng, n, spd) for n in sizes]
    Bs = [rng.standard_normal((n, nrhs)) for n in sizes]
    print(f"batched nrhs={nrhs} spd={spd}", flush=True)
    xs, status, eta, info = L.gesv_batched(As, Bs, np.full(len(sizes), spd, np.uint8))
    assert info.failed == 0, status
    for a, x, b, e in zip(As, xs, Bs, eta):
        check(a, x, b)
        assert e <= a.shape[0] * U64


def test_some_systems_need_fp64():
    """Out of FP32's range, too ill-conditioned for an FP32 factor, singular, or with a
    zero right-hand side, among ordinary systems of both kinds and all sizes."""
    from scirs_amd import linalg as L
    rng = np.random.default_rng(3)
    As, Bs, spd, singular = [], [], [], []
    for i, n in enumerate([256, 200, 130, 100, 70, 65, 64, 40, 33, 32, 20, 16, 9, 3] * 3):
        k = int(rng.integers(0, 2))
        a = system(rng, n, k)
        what = i % 5
        b = rng.standard_normal((n, 2))
        if what == 1:
            a *= 1e60
        elif what == 2 and not k:
            u, _ = np.linalg.qr(rng.standard_normal((n, n)))
            v, _ = np.linalg.qr(rng.standard_normal((n, n)))
            a = (u * np.logspace(0, 10, n)) @ v.T
        elif what == 3:
            b[:, 1] = 0.0
        elif what == 4 and not k:
            a[:, n // 2] = 0.0
            singular.append(i)
        As.append(a); Bs.append(b); spd.append(k)
    print("batched with FP64 systems", flush=True)
    xs, status, eta, info = L.gesv_batched(As, Bs, np.array(spd, np.uint8))
    assert info.failed == len(singular)
    for i, (a, x, b) in enumerate(zip(As, xs, Bs)):
        if i in singular:
            with pytest.raises(oracle.OracleError) as e:
                oracle.lu_factor(a)
            assert status[i] == e.value.code
        else:
            assert status[i] == 0
            check(a, x, b)
