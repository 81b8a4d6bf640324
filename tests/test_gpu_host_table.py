"""Host tables through kernel arguments: lengths around what one launch carries (960 words); the source is overwritten as soon
as the call returns, the GPU busy at that time."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 257, 959, 960, 961, 1920, 2000])
def test_words_arrive_and_the_source_may_go(n):
    from gcore_lowp import _abi as A
    print("[case] host table", n, flush=True)
    want = [(i * 2654435761 + n) % (1 << 32) - (1 << 31) for i in range(n)]
    src = (ctypes.c_int32 * n)(*want)
    out = torch.full((n + 1,), 7, dtype=torch.int32, device="cuda")
    busy = torch.randn(4096, 4096, device="cuda")
    busy = busy @ busy
    A.check(A.lib().lp_host_table(ctypes.addressof(src), n, out.data_ptr(), A.stream_ptr()))
    for i in range(n):
        src[i] = 0
    assert out.tolist() == want + [7]
