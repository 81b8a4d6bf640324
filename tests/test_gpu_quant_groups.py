"""The 1 x 128 quantiser where its launch changes: group counts around a workgroup's 16 (one pass), around the 2^17 from which a
workgroup makes several passes, and remainders of its 32 / 64 groups there; bit-exact against the eager oracle, and a NaN in the
last group counted once."""
import pytest
import torch

from oracle import torch_ref as T
from tests import _inputs as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("groups", [1, 15, 16, 17, 1 << 17, (1 << 17) + 1, (1 << 17) + 33, (1 << 17) + 64])
def test_group_counts(groups, dtype):
    import gcore_lowp as G
    from gcore_lowp import _abi as A, ops
    x = I.act_like(groups, 128, groups, dtype=dtype)
    print("[case] groups", groups, dtype, flush=True)
    xg = x.cuda()
    q, s = G.quant_1d(xg)
    rq, rs = T.quant_block_fp32_scale(x, (1, 128))
    assert torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s.cpu(), rs)
    q, s = G.quant_fp8_e4m3_scale_e8m0(xg.to(torch.bfloat16), (1, 128))
    rq, rs = T.quant_fp8_e4m3_scale_e8m0(x.to(torch.bfloat16), (1, 128))
    assert torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s.cpu().view(torch.uint8), rs.view(torch.uint8))
    xg[-1, 77] = float("nan")
    _, _, n = ops.quant_fp8_block(xg, (1, 128), scale_mode=A.SCALE_POW2, scale_dtype=ops.E8M0, count_nan=True)
    assert n == 1
