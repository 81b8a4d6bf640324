"""Short-K products just past a round of 256 x 256 tiles, which run on 128 x 128 ones where those fill whole rounds: against float64, with cases on
both sides of every line of the rule."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    (2409, 6528, 1152), (1665, 9216, 2688), (2305, 6912, 128), (2817, 5888, 2688), (4097, 7936, 2048),      # 128 x 128: 969, 1008, 1026 > 1024, 1058, 2046 tiles
    (1665, 9216, 2816), (4097, 7936, 2176),                                                              # K one block longer: 256-row tiles
]


@pytest.mark.parametrize("pow2", [False, True], ids=["f32scale", "e8m0scale"])
@pytest.mark.parametrize("M,N,K", CASES, ids=str)
def test_products_past_a_round(M, N, K, pow2):
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    print("[case]", (M, N, K), pow2, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + K)
    xq, wq = (torch.randn(r, K, generator=g, device="cuda").to(torch.float8_e4m3fn) for r in (M, N))
    xs, ws = (torch.randint(120, 126, s, generator=g, device="cuda", dtype=torch.uint8) for s in ((M, K // 128), (N // 128, K // 128)))
    if not pow2:
        xs, ws = (torch.pow(2.0, t.float() - 127) * 1.25 for t in (xs, ws))
    guard = 4096
    room = torch.full((M * N + guard,), float("nan"), device="cuda")
    A.check(L.lp_gemm_fp8_block(xq.data_ptr(), xs.data_ptr(), wq.data_ptr(), ws.data_ptr(), A.E8M0 if pow2 else A.F32, M, N, K, room.data_ptr(), A.F32,
                                None, 0, A.stream_ptr()))
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
