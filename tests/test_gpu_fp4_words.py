"""The fused FP4 -> FP8 conversion with two packed words per lane (aligned buffers) against the form with one (buffers off 8 and 16 bytes): the same
bytes, for odd numbers of tiles per row and edge scale bytes, from one tile to 4160 workgroups of two."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def convert(packed, scale, mode, dtype, shift, guarded=True):
    """lp_fp4_to_fp8_amax with the codes and the packed input `shift` times 4 / 8 bytes off their alignment"""
    from gcore_lowp import _abi as A
    rows, cols = packed.shape[0], packed.shape[1] * 2
    src = torch.empty(packed.numel() + 64, dtype=torch.uint8, device="cuda")
    src = src[4 * shift:4 * shift + packed.numel()].copy_(packed.flatten())
    q = torch.full((rows * cols + 64,), 77, dtype=torch.uint8, device="cuda")
    out = q[16 + 8 * shift:16 + 8 * shift + rows * cols]
    assert src.data_ptr() % 8 == 4 * shift and out.data_ptr() % 16 == 8 * shift
    s = torch.empty(rows // 128, cols // 128, dtype=torch.float32 if dtype == A.F32 else torch.uint8, device="cuda")
    A.check(A.lib().lp_fp4_to_fp8_amax(src.data_ptr(), scale.data_ptr(), rows, cols, mode, 1e-12 if mode == A.SCALE_DIV else 0.0, 0, out.data_ptr(),
                                       s.data_ptr(), dtype, None, A.stream_ptr()))
    assert not guarded or bool((q[:16 + 8 * shift] == 77).all()) and bool((q[16 + 8 * shift + rows * cols:] == 77).all())
    return out, s


@pytest.mark.parametrize("rows,cols", [(128, 128), (128, 384), (256, 256), (384, 1664), (1024, 2048), (128 * 64, 64 * 256), (128 * 64, 65 * 256)])
@pytest.mark.parametrize("edge", [False, True])
def test_two_words_a_lane(rows, cols, edge):
    from gcore_lowp import _abi as A
    g = torch.Generator(device="cuda").manual_seed(rows + cols + edge)
    packed = torch.randint(0, 256, (rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
    scale = torch.randint(100, 128, (rows, cols // 32), generator=g, device="cuda", dtype=torch.uint8)
    scale.view(rows, cols // 128, 4)[:] -= (torch.arange(cols // 128, device="cuda", dtype=torch.uint8) % 7 * 3)[None, :, None]      # no two neighbours alike
    if edge:                                   # whole super tiles take the literal path; others hold nothing but zeros
        scale[5, ::12] = 0
        scale[7, 3::8] = 254
        scale[100, 4::16] = 255
        packed[:128, :64] = 0
    for mode, dtype in ((A.SCALE_DIV, A.F32), (A.SCALE_POW2, A.E8M0), (A.SCALE_MUL, A.F32)):
        print("[case]", rows, cols, edge, mode, flush=True)
        (a, sa), (b, sb) = (convert(packed, scale, mode, dtype, shift) for shift in (0, 1))
        assert torch.equal(a, b) and torch.equal(sa.view(torch.uint8), sb.view(torch.uint8))
