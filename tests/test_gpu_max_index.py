"""rtps_max_i32, the bound check of permute and leapfrog: the maximum of the
first n entries as signed integers, at the edges of its blocks, wherever it lies;
both operators still refuse an index past their arrays."""
import numpy as np
import pytest
import torch

from enjaparticles_amd import _native as N
from enjaparticles_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 255, 256, 257, 16384, 16385, 100003])
def test_max_of_the_first_n(n):
    import ctypes as C
    rng = np.random.default_rng(n)
    host = rng.integers(-2**31, 2**31 - 1, n + 5).astype(np.int32)
    host[n:] = 2**31 - 1                       # entries past n do not count
    for at in {0, n // 2, n - 1} if n else {0}:
        v = host.copy()
        if n:
            v[:n] = np.minimum(v[:n], 1000)
            v[at] = 1001
        d = torch.from_numpy(v).cuda()
        out = C.c_int32()
        N.check(N.lib().rtps_max_i32(n, d.data_ptr(), C.byref(out), torch.cuda.current_stream().cuda_stream))
        assert out.value == (1001 if n else -2**31)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_operators_refuse_an_index_past_their_arrays(dtype):
    f4 = torch.zeros(300, 4, device="cuda")
    idx = torch.arange(300, dtype=torch.int32, device="cuda")
    idx[299] = 300
    with pytest.raises(ValueError):
        ops.permute(idx.to(dtype), f4, f4, f4)
    sp = N.SPHParams()
    with pytest.raises(ValueError):
        ops.leapfrog(f4, f4, f4, f4, idx.to(dtype), sp, 0.003, f4, f4, f4)
    ps, _, _ = ops.permute(idx, f4, f4, f4, num=299)
    assert ps.shape == (299, 4)
