"""The streaming dequantisers where a workgroup's range ends inside the tensor (512 chunks of 8 values, 1024 for large packed tensors)
and around the size where packed tensors take more per workgroup; bit-exact against the eager oracle."""
import pytest
import torch

from oracle import torch_ref as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 128), (31, 128), (32, 128), (33, 128), (65, 384), (8192, 8192), (8193, 8192)])
@pytest.mark.parametrize("fp4", [False, True], ids=["fp8", "fp4"])
def test_ragged_ends(rows, cols, fp4):
    import gcore_lowp as G
    print("[case] dequant", rows, cols, "fp4" if fp4 else "fp8", flush=True)
    g = torch.Generator().manual_seed(rows + cols)
    bn = 32 if fp4 else 128
    codes = torch.randint(0, 256, (rows, cols // 2 if fp4 else cols), generator=g, dtype=torch.int32).to(torch.uint8)
    codes = codes.view(torch.int8) if fp4 else torch.where(codes & 0x7F == 0x7F, 0, codes).to(torch.uint8).view(torch.float8_e4m3fn)
    scales = torch.randint(100, 140, (rows, cols // bn), generator=g, dtype=torch.int32).to(torch.uint8).view(torch.float8_e8m0fnu)
    got = G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(codes.cuda(), scales.cuda())
    want = T.dequant_fp4_e2m1_fp8_scale_e8m0_packed(codes, scales)
    assert torch.equal(got.cpu().view(torch.int16), want.view(torch.int16))
