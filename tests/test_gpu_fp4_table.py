"""The fused FP4 -> FP8 conversion where its two ways of building a pass's code table meet: scale bytes that reach `span` powers of
two below the tile's largest (the moved table serves 11 when the largest value is a 6, fewer otherwise), tiles whose largest
values are the small ones, all-zero blocks with scale bytes far above and below the others; every scale rule, bit-exact."""
import pytest
import torch

from oracle import torch_ref as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("span", [0, 9, 10, 11, 12, 13, 40])
@pytest.mark.parametrize("top", [1, 2, 3, 5, 7], ids=lambda c: f"code{c}")
def test_scale_spans(span, top):
    import gcore_lowp as G
    from gcore_lowp import _abi as A, ops
    print("[case] fp4 table", span, top, flush=True)
    g = torch.Generator().manual_seed(100 * span + top)
    rows, cols = 256, 384
    nib = torch.randint(0, top + 1, (rows, cols), generator=g) | (torch.randint(0, 2, (rows, cols), generator=g) << 3)
    sb = 124 - torch.randint(0, span + 1, (rows, cols // 32), generator=g)
    sb[0, ::4], nib[0, ::128] = 124, top                   # every tile has its largest value and, below it, the smallest scale
    sb[1, ::4], sb[2, 1::4], sb[3, 2::4] = 124 - span, 200, 30
    nib[2].view(-1, 32)[1::4] = 0                          # zero blocks: scale bytes that no value constrains
    nib[3].view(-1, 32)[2::4] = 8
    p = (nib[:, ::2] | (nib[:, 1::2] << 4)).to(torch.uint8).view(torch.int8)
    s = sb.to(torch.uint8).view(torch.float8_e8m0fnu)
    w = T.cast_e2m1fn_to_bf16(p, s)
    pairs = [(T.fp4_to_fp8_amax(p, s), G.fp4_to_fp8_blockwise(p.cuda(), s.cuda())),
             (T.quant_fp8_e4m3_scale_e8m0(w, (128, 128)), ops.fp4_to_fp8_amax(
                 p.view(torch.uint8).cuda(), s.cuda(), scale_mode=A.SCALE_POW2, scale_dtype=torch.float8_e8m0fnu, amax_floor=0.0)),
             (T.quantize_fp8_blockwise(w, (128, 128), scale_dtype=torch.float32), ops.fp4_to_fp8_amax(
                 p.view(torch.uint8).cuda(), s.cuda(), scale_mode=A.SCALE_MUL, scale_dtype=torch.float32, amax_floor=0.0))]
    for (rq, rs), (hq, hs) in pairs:
        assert torch.equal(hq.cpu().view(torch.uint8), rq.view(torch.uint8))
        assert torch.equal(hs.cpu().view(torch.uint8), rs.view(torch.uint8))
