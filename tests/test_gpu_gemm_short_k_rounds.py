"""Short-K products just past a round of 256 x 256 tiles, which run on 128 x 128 ones where those fill whole rounds: against float64, with cases on
both sides of every line of the rule.  Each case names the tiles it is for, and the kernels that ran are checked."""
import pytest
import torch

from tests._routes import kernels

pytestmark = pytest.mark.gpu

TILES = {"128": "gemm_asmILi128ELi128E", "256": "gemm_asmILi256ELi256E", "wide": "gemm_asm_wide", "both in one": "gemm_asm_mixed"}
CASES = [
    # (M, N, K), tiles of 128 x 128, of 256 x 256, the ones that run
    ((2409, 6528, 1152), 969, 260, "128"),
    ((2665, 6144, 2688), 1008, 264, "128"), ((2665, 6144, 2816), 1008, 264, "256"),        # 21 K blocks, 22
    ((3963, 4224, 1920), 1023, 272, "128"), ((2305, 6912, 128), 1026, 270, "256"), ((2817, 5888, 2688), 1058, 276, "256"),
    ((1665, 9216, 2688), 1008, 252, "256"),                                                # one round
    ((4097, 7936, 2048), 2046, 527, "128"), ((4097, 7936, 2176), 2046, 527, "256"), ((4097, 8064, 1152), 2079, 544, "256"),
    ((896, 18432, 1024), 1008, 288, "128"), ((896, 18432, 1536), 1008, 288, "wide"), ((1408, 11520, 1536), 990, 270, "128"), ((1408, 11520, 2048), 990, 270, "wide"),      # 256 x 288 tiles in one round
    ((2176, 14976, 1536), 1989, 531, "128"),                                               # ... in two
    # few row tiles: tiles with fp32 scales, with e8m0 scales
    ((1152, 13952, 1792), 981, 275, "128"), ((1152, 13952, 1920), 981, 275, ("128", "256")), ((1153, 12928, 1920), 1010, 255, "256"), ((1281, 11904, 1920), 1023, 282, "128"),
    ((1664, 9984, 2048), 1014, 273, ("128", "both in one")), ((1664, 9984, 2560), 1014, 273, ("128", "256")), ((1664, 9984, 2176), 1014, 273, "128"), ((1665, 9344, 2048), 1022, 259, "128"),
]


@pytest.mark.parametrize("pow2", [False, True], ids=["f32scale", "e8m0scale"])
@pytest.mark.parametrize("shape,small,big,tiles", CASES, ids=str)
def test_products_past_a_round(shape, small, big, tiles, pow2):
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    M, N, K = shape
    assert -(-M // 128) * (N // 128) == small and -(-M // 256) * -(-N // 256) == big
    print("[case]", (M, N, K), pow2, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + K)
    xq, wq = (torch.randn(r, K, generator=g, device="cuda").to(torch.float8_e4m3fn) for r in (M, N))
    xs, ws = (torch.randint(120, 126, s, generator=g, device="cuda", dtype=torch.uint8) for s in ((M, K // 128), (N // 128, K // 128)))
    if not pow2:
        xs, ws = (torch.pow(2.0, t.float() - 127) * 1.25 for t in (xs, ws))
    guard = 4096
    room = torch.full((M * N + guard,), float("nan"), device="cuda")

    def product():
        A.check(L.lp_gemm_fp8_block(xq.data_ptr(), xs.data_ptr(), wq.data_ptr(), ws.data_ptr(), A.E8M0 if pow2 else A.F32, M, N, K, room.data_ptr(), A.F32,
                                    None, 0, A.stream_ptr()))

    product()
    ran = kernels(product)
    tiles = tiles if isinstance(tiles, str) else tiles[pow2]
    # (the columns past the last whole round of 256-row tiles may be a second launch, of 128 x 128 tiles)
    assert TILES[tiles] in ran[0] and (len(ran) == 1 or tiles == "256" and len(ran) == 2 and TILES["128"] in ran[1]), ran
    out = room[:-guard].view(M, N)
    assert bool(room[-guard:].isnan().all()) and not bool(out.isnan().any())
    sx, sw = (torch.pow(2.0, t.double() - 127) if pow2 else t.double() for t in (xs, ws))
    for first in range(0, M, 1024):
        r = slice(first, min(first + 1024, M))
        exact = torch.zeros(r.stop - first, N, dtype=torch.float64, device="cuda")
        for k in range(0, K, 128):
            exact += (xq[r, k:k + 128].double() @ wq[:, k:k + 128].double().t()) * sx[r, k // 128][:, None] * sw[:, k // 128].repeat_interleave(128)[None, :]
        assert ((out[r].double() - exact).norm() / exact.norm()).item() < 4e-5      # the instruction's own sums: 1.5e-5
        assert (out[r].double() - exact).abs().max().item() < 1e-3 * exact.pow(2).mean().sqrt().item()
