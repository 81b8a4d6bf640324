"""Dense products on 128 x 160 tiles against the same products cut into column ranges that take 128 x 128 tiles: the same sums in the same order, so the
same bits, at every number of K blocks a last trip can have, at every place where a tile's columns meet the next weight scale, and where N ends inside a tile."""
import pytest
import torch

from oracle import torch_ref as T
from tests import _inputs as I

pytestmark = pytest.mark.gpu

# (M, N, K): tiles of 128 in (256, ..], of 160 at most 256; or above 512 and at most 512
CASES = [
    (1000, 5120, 2816), (1000, 4992, 2944), (1000, 4736, 2944), (900, 5120, 2176), (1024, 5120, 2560), (1000, 5120, 2688),      # one a CU; K blocks 1 .. 3 past a trip of four and none
    (256, 17408, 2816), (130, 16512, 2944), (129, 20480, 2304), (3969, 1152, 2944), (4000, 1280, 2560),     # two rows of tiles; the last of one row; few columns
    (1000, 10240, 2560), (1000, 8704, 2944), (500, 17408, 2176),                                            # two a CU
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("pow2", [False, True], ids=["f32scale", "e8m0scale"])
@pytest.mark.parametrize("M,N,K", CASES, ids=str)
def test_same_bits_as_128_wide_tiles(M, N, K, pow2, dtype):
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    print("[case]", (M, N, K), pow2, dtype, flush=True)
    quant = T.quant_fp8_e4m3_scale_e8m0 if pow2 else T.quant_block_fp32_scale
    (xq, xs), (wq, ws) = quant(I.act_like(M, K, M + K), (1, 128)), quant(I.weight_like(N, K, N, outliers=False), (128, 128))
    ops = [t.cuda().contiguous() for t in (xq, xs, wq, ws)]

    def product(first, last):
        guard = 4096
        room = torch.full((M * (last - first) + guard,), float("nan"), dtype=dtype, device="cuda")
        w, s = ops[2][first:last], ops[3][first // 128:last // 128]
        A.check(L.lp_gemm_fp8_block(ops[0].data_ptr(), ops[1].data_ptr(), w.data_ptr(), s.data_ptr(), A.E8M0 if pow2 else A.F32, M, last - first, K,
                                    room.data_ptr(), A.BF16 if dtype == torch.bfloat16 else A.F32, None, 0, A.stream_ptr()))
        assert bool(room[-guard:].isnan().all())
        return room[:-guard].view(M, last - first)

    got = product(0, N)
    # column ranges of at most 255 tiles, alike: whole columns of tiles, more than the decode kernels take in slices of 128 rows
    rows, columns = -(-M // 128), N // 128
    parts = -(-columns // max(1, 255 // rows))
    for i in range(parts):
        first, last = (columns * j // parts * 128 for j in (i, i + 1))
        want = product(first, last)
        bad = (got[:, first:last] != want).nonzero()
        assert not len(bad), (first, last, len(bad), bad[:4].tolist())
