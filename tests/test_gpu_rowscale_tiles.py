"""The row-scaled grouped GEMM on both tile sizes of its loop (256 x 256 tiles need at least 256 of them and at most a tenth beyond
the matrix): matrices that end inside a tile, three K blocks up to two trips of four and each remainder, an unaligned scale
table (an odd number of blocks in front).  Bound as in tests/test_gpu_any_k.py."""
import pytest
import torch

from tests.test_gpu_any_k import close, deq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(384, 640), (2048, 2176), (2304, 4096)], ids=["tiles128", "tiles256_ragged", "tiles256"])
def test_problems_of_any_length(M, N):
    import gcore_lowp as G
    k_blocks = [3, 9, 1, 4, 5, 2, 8, 6, 7, 0, 11]
    g = torch.Generator(device="cuda").manual_seed(M)
    ops = []
    for kb in k_blocks:
        if kb:
            a = torch.randn(M, kb * 128, generator=g, device="cuda", dtype=torch.bfloat16)
            b = torch.randn(N, kb * 128, generator=g, device="cuda", dtype=torch.bfloat16) * 0.05
            ops.append(G.quant_fp8_e4m3_scale_e8m0(a, (1, 128)) + G.quant_fp8_e4m3_scale_e8m0(b, (1, 128)))
        else:
            ops.append(None)
    flat = [torch.cat([o[i].view(torch.uint8).flatten() for o in ops if o]) for i in range(4)]
    out = torch.full((len(k_blocks), M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    G.gemm_fp8_rowscale_grouped(*flat, k_blocks, M, N, out)
    for e, o in enumerate(ops):
        if o is None:
            assert not out[e].any()
        else:
            close(out[e], deq(o[0], o[1], 1) @ deq(o[2], o[3], 1).t(), ("rowscale", M, N, k_blocks[e]))
