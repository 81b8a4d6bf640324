"""Row-scaled problems of two K blocks, walked in strips of column tiles: one tile, strips that end in the matrix (9, 17 tiles),
row panels that do not fill a group of eight, bf16 and fp32 results, problems out of order, a single problem without a table,
and an entry of another size, whose slot stays as it was.  Few problems: strips cut shorter than eight tiles (one tile, two, uneven
last ones) and dealt in pieces smaller than eight.  Bound as in tests/test_gpu_any_k.py."""
import pytest
import torch

from tests.test_gpu_any_k import close, deq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("M,N,E", [(128, 128, 1), (1152, 1152, 3), (384, 2176, 2), (2048, 1024, 5), (128, 1024, 1), (1408, 1024, 1), (256, 1664, 2), (1024, 2048, 4)])
def test_two_k_blocks(M, N, E, dtype):
    import gcore_lowp as G
    g = torch.Generator(device="cuda").manual_seed(M + N)
    ops = [G.quant_fp8_e4m3_scale_e8m0(torch.randn(M, 256, generator=g, device="cuda", dtype=torch.bfloat16), (1, 128))
           + G.quant_fp8_e4m3_scale_e8m0(torch.randn(N, 256, generator=g, device="cuda", dtype=torch.bfloat16) * 0.05, (1, 128)) for _ in range(E)]
    flat = [torch.cat([o[i].view(torch.uint8).flatten() for o in ops]) for i in range(4)]
    out = torch.full((E, M, N), float("nan"), dtype=dtype, device="cuda")
    print("[case]", M, N, E, dtype, flush=True)
    G.gemm_fp8_rowscale_grouped(*flat, [2] * E, M, N, out)
    for e, o in enumerate(ops):
        close(out[e], deq(o[0], o[1], 1) @ deq(o[2], o[3], 1).t(), ("strip", M, N, e))
    one = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    G.gemm_fp8_rowscale(*(f[:f.numel() // E] for f in flat), M, N, 256, one)
    assert torch.equal(one, out[0])


def test_entry_of_another_size_writes_nothing():
    from gcore_lowp import _abi as A
    M = N = 256
    a = torch.zeros(3 * M * 256, dtype=torch.uint8, device="cuda")
    s = torch.full((3 * M * 2,), 127, dtype=torch.uint8, device="cuda")
    out = torch.full((3, M, N), 5.0, dtype=torch.bfloat16, device="cuda")
    table = torch.tensor([[0, 2, 0, 0], [1, 1, 2, 0], [2, 2, 4, 0]], dtype=torch.int32, device="cuda")
    A.check(A.lib().lp_gemm_fp8_rowscale_grouped(a.data_ptr(), s.data_ptr(), a.data_ptr(), s.data_ptr(), A.E8M0, table.data_ptr(), 3, 2, 2,
                                                 M, N, out.data_ptr(), A.BF16, A.stream_ptr()))
    assert not out[0].any() and not out[2].any() and bool((out[1] == 5.0).all())
