"""The forms of the fused FP4 -> FP8 conversion with two words a lane (two scale tiles to a workgroup, scale bytes handed round or loaded one by one; four tiles)
against the form with one word a lane (buffers off their alignment): the same bytes on both sides of every size where the form changes, where the last
workgroup of a row has one, two, three or four tiles, with edge scale bytes in any of them, and with scales that start anywhere.  Each case names the form it is for."""
import pytest
import torch

from tests._routes import kernels
from tests.test_gpu_fp4_words import convert

pytestmark = pytest.mark.gpu

FORMS = {"handed": "ELb0ELi256ELi2ELi2ELb0E", "bytes": "ELb0ELi256ELi2ELi2ELb1E", "four": "ELb0ELi512ELi2ELi4ELb0E",
         "one word": "ELb0ELi256ELi1ELi2ELb1ELb1E", "one word, many": "ELb0ELi256ELi1ELi2ELb1ELb0E"}
CASES = [
    # (rows of tiles, tiles a row), form
    ((768, 2), "handed"), ((769, 2), "bytes"), ((1280, 2), "bytes"), ((1281, 2), "handed"), ((600, 1), "handed"),      # four tiles would leave half of them empty
    ((384, 3), "handed"), ((385, 3), "four"), ((384, 4), "handed"), ((385, 4), "four"),
    ((300, 5), "bytes"),                                                                                              # a quarter empty
    ((192, 7), "handed"), ((193, 7), "four"), ((192, 8), "handed"), ((193, 8), "four"), ((224, 8), "four"), ((225, 8), "bytes"), ((320, 8), "bytes"), ((321, 8), "four"),
    ((64, 16), "handed"), ((65, 16), "bytes"), ((96, 16), "bytes"), ((97, 16), "four"), ((89, 18), "bytes"),
    ((30, 33), "handed"), ((31, 33), "bytes"), ((45, 33), "bytes"), ((46, 33), "four"), ((30, 34), "handed"), ((45, 34), "bytes"), ((46, 34), "four"), ((43, 35), "four"),
]


def check(packed, scale, modes, form):
    for mode, dtype in modes:
        (a, sa), (b, sb) = (convert(packed, scale, mode, dtype, shift) for shift in (0, 1))
        assert torch.equal(a, b) and torch.equal(sa.view(torch.uint8), sb.view(torch.uint8))
    pairs = packed.shape[0] // 128 * -(-packed.shape[1] // 128)
    for shift, wanted in ((0, form), (1, "one word, many" if pairs > 1280 else "one word")):
        ran = kernels(lambda: convert(packed, scale, *modes[0], shift, False))
        assert [FORMS[wanted] in n for n in ran if "fp4_amax" in n] == [True], (wanted, ran)


@pytest.mark.parametrize("size,form", CASES, ids=str)
@pytest.mark.parametrize("edge", [False, True])
def test_forms_give_the_same_bytes(size, form, edge):
    from gcore_lowp import _abi as A
    rows, tiles = 128 * size[0], size[1]
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
    print("[case]", rows, cols, edge, form, flush=True)
    check(packed, scale, ((A.SCALE_DIV, A.F32), (A.SCALE_POW2, A.E8M0), (A.SCALE_MUL, A.F32)), form)


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("size,form", [((3, 5), "handed"), ((65, 16), "bytes"), ((46, 34), "four")], ids=str)
def test_scales_off_their_alignment(size, form, offset):
    """Scale bytes that start anywhere: the same kernels, the same result."""
    from gcore_lowp import _abi as A
    g = torch.Generator(device="cuda").manual_seed(3)
    rows, cols = 128 * size[0], 128 * size[1]
    packed = torch.randint(0, 256, (rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
    flat = torch.randint(117, 128, (rows * cols // 32 + 4,), generator=g, device="cuda", dtype=torch.uint8)
    scale = flat[offset:offset + rows * cols // 32].view(rows, cols // 32)
    assert scale.data_ptr() % 4 == offset
    print("[case] scale offset", offset, size, flush=True)
    check(packed, scale, ((A.SCALE_DIV, A.F32),), form)
    a, sa = convert(packed, scale, A.SCALE_DIV, A.F32, 0)
    b, sb = convert(packed, scale.clone(), A.SCALE_DIV, A.F32, 0)
    assert torch.equal(a, b) and torch.equal(sa, sb)
