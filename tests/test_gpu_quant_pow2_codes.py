"""Power-of-two scales on bf16 input: the conversion that divides by the scale itself, over every finite bf16 value under every scale that
value can meet, and the tile counts at which the 128 x 128 launch changes.  Bit-exact; the expected codes are torch's own
cast of the exact quotient."""
import pytest
import torch

from oracle import torch_ref as T
from tests import _inputs as I

pytestmark = pytest.mark.gpu

EXPONENTS = list(range(-126, 120))


def _patterns(e):
    """Every finite bf16 value, those over 448 * 2^e replaced by it: 512 groups of 128, the largest quotient 448 in each."""
    x = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    top = 448.0 * 2.0 ** e
    x = torch.where(x.float().abs() <= top, x.float(), torch.full((), top)).to(torch.bfloat16).view(512, 128).clone()
    x[:, 5] = top
    return x


def _want(x, e):
    return (x.double() * 2.0 ** -e).float().to(torch.float8_e4m3fn).view(torch.uint8)


@pytest.fixture(scope="module")
def every():
    x = torch.cat([_patterns(e) for e in EXPONENTS])
    return x, torch.cat([_want(x[512 * i:512 * (i + 1)], e) for i, e in enumerate(EXPONENTS)])


def _scales(s):
    return (s.cpu().view(torch.uint8).to(torch.int32) - 127).flatten()


@pytest.mark.parametrize("copies", [1, 4], ids=["few tiles", "runs of tiles"])
def test_every_value_in_tiles(every, copies):
    import gcore_lowp as G
    x, want = (t.cuda().repeat(copies, 1) for t in every)
    print("[case] tiles", x.shape[0] // 128, flush=True)
    q, s = G.quant_fp8_e4m3_scale_e8m0(x)
    assert torch.equal(q.view(torch.uint8), want)
    assert torch.equal(_scales(s), torch.tensor(EXPONENTS, dtype=torch.int32).repeat_interleave(4).repeat(copies))


def test_every_value_in_rows_and_columns(every):
    """The rows' and the columns' quantisation of a training step (a column's groups are the patterns; a row's are whatever lies side by side)."""
    from gcore_lowp import _abi as A
    x, want = every
    n = x.shape[0]
    xt = x.t().contiguous().cuda()
    print("[case] columns", n, flush=True)
    offs = torch.tensor([0, 128], dtype=torch.int32, device="cuda")
    q, qT = torch.empty(128, n, dtype=torch.uint8, device="cuda"), torch.empty(n, 128, dtype=torch.uint8, device="cuda")
    s, sT = torch.empty(128, n // 128, dtype=torch.uint8, device="cuda"), torch.empty(n, dtype=torch.uint8, device="cuda")
    A.check(A.lib().lp_quant_fp8_row_colwise_t(xt.data_ptr(), A.BF16, 128, n, offs.data_ptr(), 1, 1, 128, q.data_ptr(), s.data_ptr(), qT.data_ptr(),
                                               sT.data_ptr(), A.E8M0, A.stream_ptr()))
    assert torch.equal(qT.cpu(), want)
    assert torch.equal(_scales(sT), torch.tensor(EXPONENTS, dtype=torch.int32).repeat_interleave(512))
    rq, rs = T.quant_fp8_e4m3_scale_e8m0(x.t().contiguous(), (1, 128))
    assert torch.equal(q.cpu(), rq.view(torch.uint8)) and torch.equal(s.cpu(), rs.view(torch.uint8))


@pytest.mark.parametrize("mode", ["pow2", "div"])
@pytest.mark.parametrize("rows,cols", [(128, 128 * 3071), (128, 128 * 3072), (128 * 3073, 128), (128 * 61, 128 * 51), (128 * 7, 128 * 439)], ids=str)
def test_tile_counts(rows, cols, mode):
    import gcore_lowp as G
    x = I.weight_like(rows, cols, rows + cols).to(torch.bfloat16)
    print("[case]", rows, cols, mode, flush=True)
    xg = x.cuda()
    q, s = G.quant_fp8_e4m3_scale_e8m0(xg) if mode == "pow2" else G.quant_2d(xg)
    rq, rs = T.quant_fp8_e4m3_scale_e8m0(x) if mode == "pow2" else T.quant_block_fp32_scale(x, (128, 128))
    assert torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s.cpu().view(torch.uint8), rs.view(torch.uint8))


def test_nan_in_the_last_tile_of_a_run():
    from gcore_lowp import _abi as A, ops
    x = torch.ones(128 * 3079, 128, dtype=torch.bfloat16, device="cuda")
    x[-1, -1] = float("nan")
    print("[case] nan", flush=True)
    _, _, n = ops.quant_fp8_block(x, (128, 128), scale_mode=A.SCALE_POW2, scale_dtype=ops.E8M0, count_nan=True)
    assert n == 1
