"""A batch whose workspace exceeds the limit (SCIRS_GPU_BATCH_WORK_MB) runs in chunks: the
same solutions and states bit for bit, and no more memory."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_chunks_give_the_same_solutions(monkeypatch):
    from scirs_amd import linalg as L
    rng = np.random.default_rng(8)
    As, Bs, spd = [], [], []
    for i in range(150):
        n = int(rng.integers(1, 257))
        g = rng.standard_normal((n, n))
        k = int(rng.integers(0, 2))
        a = g @ g.T / n + np.eye(n) if k else g + 2.0 * np.diag(rng.choice([-1.0, 1.0], n))
        if i % 7 == 0:
            a = a * 1e60                    # out of FP32's range: the FP64 launch
        if i % 31 == 5 and not k:
            a[:, n // 2] = 0.0              # singular
        As.append(a)
        Bs.append(rng.standard_normal((n, 1 + i % 5)))
        spd.append(k)
    spd = np.array(spd, np.uint8)
    monkeypatch.delenv("SCIRS_GPU_BATCH_WORK_MB", raising=False)
    want, status, eta, _ = L.gesv_batched(As, Bs, spd)
    for mb in ("1", "3", "1000000"):
        monkeypatch.setenv("SCIRS_GPU_BATCH_WORK_MB", mb)
        print(f"batch in chunks of {mb} MiB", flush=True)
        got, st, et, info = L.gesv_batched(As, Bs, spd)
        assert np.array_equal(st, status) and np.array_equal(et, eta)
        for x, y, s in zip(got, want, status):
            if s == 0:
                assert np.array_equal(x, y)


MEMORY = r'''
import sys
sys.path.insert(0, ROOT)
import numpy as np
import torch
from scirs_amd import linalg as L
count, n = 2000000, 2
a = torch.eye(n, dtype=torch.float64, device="cuda").mul_(3.0).repeat(count, 1, 1).reshape(-1)
b = torch.ones(count * n, dtype=torch.float64, device="cuda")
x = torch.empty_like(b)
off = np.arange(count, dtype=np.int64)
one = np.ones(count, np.int32)
L.gesv_batched_dev(one[:1] * n, one[:1], off[:1], off[:1], a, b, x)   # the library's own buffers
torch.cuda.synchronize()
free = torch.cuda.mem_get_info()[0]
status, _, info = L.gesv_batched_dev(one * n, one, off * n * n, off * n, a, b, x)
print("GB", (free - torch.cuda.mem_get_info()[0]) / 1e9, "failed", info.failed, bool((x == 1.0 / 3.0).all()))
'''


def test_small_systems_do_not_take_memory_without_bound():
    """Two million systems of two rows: 10 GB if each had a workspace of its own."""
    env = {k: v for k, v in os.environ.items() if k != "SCIRS_GPU_BATCH_WORK_MB"}
    out = subprocess.run([sys.executable, "-c", MEMORY.replace("ROOT", repr(ROOT))], env=env, capture_output=True,
                         text=True, timeout=110)
    print(out.stdout[-500:], out.stderr[-500:])
    assert out.returncode == 0
    words = out.stdout.split()
    assert words[words.index("failed") + 1] == "0" and words[-1] == "True"
    assert float(words[words.index("GB") + 1]) <= 9.2     # 8 GiB and the per-system arrays
