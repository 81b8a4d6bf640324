"""The fused FP4 -> FP8 conversion with four scale tiles to a workgroup (more than 512 pairs of tiles) against the form with one word a lane
(buffers off their alignment): the same bytes where the last workgroup of a row has one, two or three tiles, around the size where the
form changes, and with edge scale bytes in any of the four tiles."""
import pytest
import torch

from tests._routes import kernels
from tests.test_gpu_fp4_words import convert

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,tiles", [(128 * 128, 8), (128 * 129, 8), (128 * 260, 3), (128 * 140, 7), (128 * 33, 33), (128 * 30, 34), (128 * 600, 1), (128 * 300, 5)], ids=str)
@pytest.mark.parametrize("edge", [False, True])
def test_four_tiles_a_workgroup(rows, tiles, edge):
    from gcore_lowp import _abi as A
    cols = 128 * tiles
    g = torch.Generator(device="cuda").manual_seed(rows + cols + edge)
    packed = torch.randint(0, 256, (rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
    scale = torch.randint(60, 128, (rows, cols // 32), generator=g, device="cuda", dtype=torch.uint8)      # small scales: both ways of building a code table
    if edge:
        scale[5, ::12] = 0
        scale[300, 4 * tiles - 1] = 254                    # the last tile of a row
        scale[128 * 7 + 100, 4::16] = 255
        packed[128:256] = 0                                # tiles of zeros beside others
        packed[128:256, :64] = 0x12
    for mode, dtype in ((A.SCALE_DIV, A.F32), (A.SCALE_POW2, A.E8M0), (A.SCALE_MUL, A.F32)):
        print("[case]", rows, cols, edge, mode, flush=True)
        (a, sa), (b, sb) = (convert(packed, scale, mode, dtype, shift) for shift in (0, 1))
        assert torch.equal(a, b) and torch.equal(sa.view(torch.uint8), sb.view(torch.uint8))


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("rows,tiles,kernel", [(384, 5, "ELb0ELi256ELi2ELi2E"), (128 * 31, 34, "ELb0ELi512ELi2ELi4E")], ids=["two tiles", "four tiles"])
def test_scales_off_their_alignment(rows, tiles, kernel, offset):
    """Scale bytes that start anywhere: the same kernel, the same result."""
    from gcore_lowp import _abi as A
    g = torch.Generator(device="cuda").manual_seed(3)
    cols = 128 * tiles
    packed = torch.randint(0, 256, (rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
    flat = torch.randint(117, 128, (rows * cols // 32 + 4,), generator=g, device="cuda", dtype=torch.uint8)
    scale = flat[offset:offset + rows * cols // 32].view(rows, cols // 32)
    assert scale.data_ptr() % 4 == offset
    print("[case] scale offset", offset, rows, cols, flush=True)
    a, sa = convert(packed, scale, A.SCALE_DIV, A.F32, 0)
    b, sb = convert(packed, scale.clone(), A.SCALE_DIV, A.F32, 0)
    c, sc = convert(packed, scale, A.SCALE_DIV, A.F32, 1)
    assert torch.equal(a, b) and torch.equal(sa, sb) and torch.equal(a, c) and torch.equal(sa, sc)
    ran = kernels(lambda: convert(packed, scale, A.SCALE_DIV, A.F32, 0, guarded=False))
    assert [kernel in n for n in ran if "fp4_amax" in n] == [True], ran
