"""LU panels across a restart of their exchange tags (2047 panels a count): the same
matrix gives the same factors, bit for bit, before and after."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_factors_across_a_restart(dtype):
    import torch  # noqa: F401
    from scirs_amd import linalg as L
    rng = np.random.default_rng(5)
    sizes = (1500, 5000) if dtype == np.float64 else (1500, 9000)
    mats = [rng.standard_normal((n, 1500)).astype(dtype) for n in sizes]
    first = [L.getrf(a)[:2] for a in mats]
    for k in range(40):                                  # 62 (f32) or 78 of its panels exchange by tags
        print(f"restart {dtype.__name__} round {k}", flush=True)
        for a, (lu, perm) in zip(mats, first):
            lu2, perm2, _ = L.getrf(a)
            assert np.array_equal(perm, perm2) and np.array_equal(lu, lu2)
