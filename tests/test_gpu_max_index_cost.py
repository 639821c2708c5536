"""The index check of permute and leapfrog costs no more than torch's maximum and its
copy to the host, which it stands in for, from small to the largest systems."""
import ctypes as C
import time

import pytest
import torch

from enjaparticles_amd import _native as N

pytestmark = pytest.mark.gpu


def _best(f):
    out = []
    for _ in range(30):
        torch.cuda.synchronize()
        t = time.perf_counter()
        f()
        out.append(time.perf_counter() - t)
    return sorted(out)[len(out) // 4]


@pytest.mark.parametrize("n", [1000, 50021, 1_000_000, 4_000_037])
def test_cost_against_torch(cuda, n):
    v = torch.randperm(n, device=cuda, dtype=torch.int32)
    out = C.c_int32()
    stream = torch.cuda.current_stream().cuda_stream
    ours = _best(lambda: N.check(N.lib().rtps_max_i32(n, v.data_ptr(), C.byref(out), stream)))
    assert out.value == n - 1
    torchs = _best(lambda: int(v.max().item()))
    print(f"{n}: {1e6 * ours:.1f} us, torch {1e6 * torchs:.1f} us")
    assert ours < 1.1 * torchs + 2e-6
