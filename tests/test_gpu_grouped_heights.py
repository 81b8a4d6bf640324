"""Grouped products whose row counts the host knows choose between tiles of 128 x 128 and of two heights by the tiles there are; with the offsets in
device memory the choice is by rows and experts alone.  Where the two differ, both give the same bits: a sum over K is the matrix instruction's, block by block, in either."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = {
    # rows per expert, N, K: what the host's rule takes, the other kernel being the device's
    "short_k_128": ([300] * 10 + [80] * 10, 3328, 1664),
    "one_tile_a_cu_128": ([2, 0, 0, 0, 0, 0, 0, 0, 0, 0] * 15, 1280, 3840),
    "a_few_in_a_second_round_128": ([3, 0, 0] * 46, 1408, 3456),
    "one_round_two_heights": ([200] * 3 + [56] * 9, 4608, 2816),
    "more_than_three_a_cu_two_heights": ([500] * 12 + [513], 2048, 4224),
}


@pytest.mark.parametrize("name", CASES)
def test_rows_known_to_the_host_give_the_same_bits(name):
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    splits, N, K = CASES[name]
    E, M = len(splits), sum(splits)
    offsets = [sum(splits[:e]) for e in range(E + 1)]
    print("[case]", name, E, M, N, K, flush=True)
    g = torch.Generator(device="cuda").manual_seed(E)
    xq, wq = (torch.randn(r, K, generator=g, device="cuda").to(torch.float8_e4m3fn) for r in (M, E * N))
    xs, ws = (torch.randint(120, 126, s, generator=g, device="cuda", dtype=torch.uint8) for s in ((M, K // 128), (E * N // 128, K // 128)))
    ops = (xq.data_ptr(), xs.data_ptr(), wq.data_ptr(), ws.data_ptr(), A.E8M0)
    out = [torch.full((M, N), float("nan"), device="cuda") for _ in range(2)]
    on_device = torch.tensor(offsets, dtype=torch.int32, device="cuda")
    A.check(L.lp_gemm_fp8_grouped(*ops, on_device.data_ptr(), E, M, N, K, out[0].data_ptr(), A.F32, A.stream_ptr()))
    on_host = (ctypes.c_int32 * (E + 1))(*offsets)
    A.check(L.lp_gemm_fp8_grouped_rows(*ops, ctypes.addressof(on_host), E, M, N, K, out[1].data_ptr(), A.F32, A.stream_ptr()))
    assert torch.equal(out[0], out[1])                          # NaN, i.e. an element left out, is equal to nothing
    e = max(range(E), key=lambda i: splits[i])                   # and the longest expert's against float64
    r = slice(offsets[e], offsets[e + 1])
    exact = torch.zeros(splits[e], N, dtype=torch.float64, device="cuda")
    for k in range(0, K, 128):
        part = xq[r, k:k + 128].double() @ wq[e * N:(e + 1) * N, k:k + 128].double().t()
        scale = torch.pow(2.0, xs[r, k // 128].double() - 127)[:, None] * torch.pow(2.0, ws[e * N // 128:(e + 1) * N // 128, k // 128].double() - 127).repeat_interleave(128)
        exact += part * scale
    assert ((out[1][r].double() - exact).norm() / exact.norm()).item() < 4e-5      # the instruction's own sums: 1.5e-5
