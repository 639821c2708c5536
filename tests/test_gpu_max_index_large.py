"""rtps_max_i32 at the largest counts, where the index of the kernel's last round
passes 2^31: the maximum may lie in the last entry, and nothing past the array is
read (the entries after the counted ones are larger)."""
import ctypes as C

import pytest
import torch

from enjaparticles_amd import _native as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2**31 - 16384, 2**31 - 16383, 2**31 - 1])
def test_max_of_counts_near_2_to_31(cuda, n):
    v = torch.full((2**31 + 64,), -5, dtype=torch.int32, device=cuda)
    v[n:] = 2**31 - 1
    out = C.c_int32()
    for at in (0, n // 2, n - 1):
        v[at] = 7
        N.check(N.lib().rtps_max_i32(n, v.data_ptr(), C.byref(out), torch.cuda.current_stream().cuda_stream))
        assert out.value == 7
        v[at] = -5
    N.check(N.lib().rtps_max_i32(n, v.data_ptr(), C.byref(out), torch.cuda.current_stream().cuda_stream))
    assert out.value == -5
    del v
    torch.cuda.empty_cache()
