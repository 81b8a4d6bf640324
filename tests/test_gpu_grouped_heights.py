"""Grouped products whose row counts the host knows choose between tiles of 128 x 128 and of two heights by the tiles there are; with the offsets in
device memory the choice is by rows and experts alone.  The cases are one or two for every line of the host's rule; each names the kernels that the two calls are to
take, which is checked.  Both give the same bits: a sum over K is the matrix instruction's, block by block, in either."""
import ctypes

import pytest
import torch

from tests._routes import kernels

pytestmark = pytest.mark.gpu

KERNELS = {"128": "gemm_asm_groupedILi128ELi128E", "two": "gemm_asm_grouped_mixed"}
CASES = {
    # rows per expert, N, K, tiles of 128 x 128 and of both heights, what the host's rule takes, what the device's
    "one_tile_a_cu": ([2] + [0] * 9, 15, 1280, 3840, 150, 75, "128", "two"),
    "second_round": ([3, 0, 0], 46, 1408, 3456, 506, 276, "128", "two"),
    "tall_experts": ([100] * 10 + [200] * 10 + [0] * 64, 1, 1408, 3200, 330, 120, "128", "two"),
    "tall_experts_beside_streams": ([40] * 21 + [176] * 2, 1, 1408, 3200, 275, 138, "two", "128"),
    "tall_and_short_of_one_expert": ([40] * 21 + [300] * 2 + [0] * 60, 1, 1408, 3200, 297, 150, "128", "two"),
    "two_a_cu_short_k": ([9, 0, 0], 46, 1280, 2432, 460, 230, "128", "two"),
    "two_a_cu_20_blocks": ([9] * 33, 1, 1536, 2560, 396, 198, "two", "128"),
    "two_a_cu_streams": ([6] * 35 + [0] * 3, 1, 1408, 3840, 385, 210, "two", "128"),
    "one_round": ([200] * 3 + [56] * 9, 1, 4608, 2816, 540, 216, "two", "128"),
    "half_a_second_round": ([7, 0], 64, 1408, 3200, 704, 384, "128", "two"),
    "half_a_second_round_36_blocks": ([24], 42, 2048, 4608, 672, 336, "128", "128"),
    "half_a_second_round_37_blocks": ([24], 42, 2048, 4736, 672, 336, "two", "128"),
    "more_of_a_second_round_32_blocks": ([24] * 48 + [0] * 16, 1, 2048, 4096, 768, 384, "128", "two"),
    "more_of_a_second_round_33_blocks": ([24], 48, 2048, 4224, 768, 384, "two", "128"),
    "short_k": ([300] * 10 + [80] * 10, 1, 3328, 1664, 1040, 390, "128", "two"),
    "short_k_of_20_blocks": ([5] * 193 + [0] * 107, 1, 512, 2560, 772, 386, "128", "two"),
    "short_k_two_full_rounds": ([64] * 12 + [200] * 3 + [300] * 3, 1, 6144, 1536, 1296, 504, "two", "two"),
    "short_k_two_rounds_14_blocks": ([38], 28, 3840, 1792, 840, 420, "two", "two"),
    "short_k_two_rounds_13_blocks": ([38], 28, 3840, 1664, 840, 420, "128", "two"),
    "short_k_400_tiles": ([64], 50, 2048, 2048, 800, 400, "128", "two"),
    "short_k_408_tiles": ([64], 51, 2048, 2048, 816, 408, "two", "two"),
    "short_k_two_rounds_for_four": ([254], 74, 1408, 1280, 1628, 444, "two", "two"),
    "short_k_two_rounds_for_three": ([254], 69, 1408, 1280, 1518, 414, "128", "two"),
    "more_than_three_a_cu": ([300] * 5 + [640] * 8, 1, 2048, 4224, 880, 272, "two", "128"),
    "streams_of_a_long_k": ([3] * 43 + [0] * 30, 1, 1536, 5504, 516, 258, "two", "128"),
    "streams_of_a_short_k": ([300] * 6 + [10] * 38 + [0] * 56, 1, 1280, 1024, 560, 250, "128", "two"),
    "by_rows": ([150] * 60, 1, 1024, 1024, 960, 240, "two", "two"),
    # the order of the XCDs: few tall tiles, few flat ones, both, and few with a long K
    "few_tall": ([8] * 296 + [300] * 4, 1, 512, 1024, 1232, 608, "128", "two"),
    "few_flat": ([256] * 140 + [50] * 8, 1, 512, 1024, 1152, 296, "128", "two"),
    "both": ([40, 200] * 70, 1, 512, 1024, 840, 280, "128", "two"),
    "few_tall_long_k": ([8] * 100 + [300] * 2, 1, 1280, 4224, 1060, 520, "two", "two"),
}


@pytest.mark.parametrize("name", CASES)
def test_rows_known_to_the_host_give_the_same_bits(name):
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    splits, times, N, K, narrow, wide, host, device = CASES[name]
    splits = splits * times
    E, M = len(splits), sum(splits)
    assert sum(-(-r // 128) for r in splits) * (N // 128) == narrow and sum(-(-r // 256) for r in splits) * -(-N // 256) == wide
    offsets = [sum(splits[:e]) for e in range(E + 1)]
    print("[case]", name, E, M, N, K, flush=True)
    g = torch.Generator(device="cuda").manual_seed(E)
    xq, wq = (torch.randn(r, K, generator=g, device="cuda").to(torch.float8_e4m3fn) for r in (M, E * N))
    xs, ws = (torch.randint(120, 126, s, generator=g, device="cuda", dtype=torch.uint8) for s in ((M, K // 128), (E * N // 128, K // 128)))
    ops = (xq.data_ptr(), xs.data_ptr(), wq.data_ptr(), ws.data_ptr(), A.E8M0)
    out = [torch.full((M, N), float("nan"), device="cuda") for _ in range(2)]
    on_device = torch.tensor(offsets, dtype=torch.int32, device="cuda")
    on_host = (ctypes.c_int32 * (E + 1))(*offsets)
    calls = ((device, lambda: A.check(L.lp_gemm_fp8_grouped(*ops, on_device.data_ptr(), E, M, N, K, out[0].data_ptr(), A.F32, A.stream_ptr()))),
             (host, lambda: A.check(L.lp_gemm_fp8_grouped_rows(*ops, ctypes.addressof(on_host), E, M, N, K, out[1].data_ptr(), A.F32, A.stream_ptr()))))
    for wanted, call in calls:
        call()
        ran = kernels(call)
        assert len(ran) == 1 and KERNELS[wanted] in ran[0], (wanted, ran)
    assert torch.equal(out[0], out[1])                          # NaN, i.e. an element left out, is equal to nothing
    # and the longest expert's and the last one's against float64
    for e in {max(range(E), key=lambda i: splits[i]), max(i for i in range(E) if splits[i])}:
        r = slice(offsets[e], offsets[e + 1])
        exact = torch.zeros(splits[e], N, dtype=torch.float64, device="cuda")
        for k in range(0, K, 128):
            part = xq[r, k:k + 128].double() @ wq[e * N:(e + 1) * N, k:k + 128].double().t()
            scale = torch.pow(2.0, xs[r, k // 128].double() - 127)[:, None] * torch.pow(2.0, ws[e * N // 128:(e + 1) * N // 128, k // 128].double() - 127).repeat_interleave(128)
            exact += part * scale
        assert ((out[1][r].double() - exact).norm() / exact.norm()).item() < 4e-5      # the instruction's own sums: 1.5e-5
