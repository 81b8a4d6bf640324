"""Both quantisations of an expert-grouped tensor from one read: the bytes of the two separate quantisers, for experts without
rows, of one row, around a block of 128 and of several, one and several column blocks, rows of zeros, of subnormals and of the
largest values, and rows and columns that hold an infinity or a NaN."""
import importlib

import pytest
import torch

from tests import _inputs as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad_rows", [128, 512])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("cols", [128, 1152])
def test_bytes_of_the_two_quantisers(cols, dtype, pad_rows):
    M = importlib.import_module("gcore_lowp.grouped_gemm_fp8")
    m_splits = [0, 1, 127, 128, 0, 129, 7, 8, 9, 300]
    rows = sum(m_splits)
    x = I.act_like(rows, cols, cols, dtype=dtype)
    big = torch.finfo(dtype).max
    x[3], x[4], x[5], x[6] = 0.0, x[4] * 1e-39, big, -big
    x[10, 5], x[140, 127], x[141, 0], x[rows - 1, cols - 1] = float("nan"), float("inf"), float("-inf"), float("nan")
    x[200, :64] = 1e-30
    xg = x.cuda()
    offs = M._offsets(m_splits, xg.device)
    print("[case]", cols, dtype, pad_rows, flush=True)
    q, s, qt, st, nblk = M._quant_rows_and_columns(xg, offs, m_splits, pad_rows)
    wq, ws = M._quant_pow2(xg, (1, 128))
    wqt, wst, wblk = M.quant_fp8_colwise_t(xg, offs, m_splits, pad_rows)
    assert nblk == wblk
    for got, want in ((q, wq), (s, ws), (qt, wqt), (st, wst)):
        assert got.shape == want.shape and torch.equal(got.view(torch.uint8), want.view(torch.uint8))


def test_misaligned_and_strided_inputs_take_the_separate_quantisers():
    M = importlib.import_module("gcore_lowp.grouped_gemm_fp8")
    m_splits = [70, 130]
    base = I.act_like(201, 256, 1).cuda()
    for xg in (base.flatten()[3:3 + 200 * 256].view(200, 256), base[:200].t().contiguous().t()):
        offs = M._offsets(m_splits, xg.device)
        got = M._quant_rows_and_columns(xg, offs, m_splits, 128)
        want = M._quant_rows_and_columns(xg.clone(memory_format=torch.contiguous_format), offs, m_splits, 128)
        for a, b in zip(got[:4], want[:4]):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
