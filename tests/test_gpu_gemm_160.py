"""Dense products on 128 x 160 tiles against the same products cut into column ranges that take 128 x 128 tiles: the same sums in the same order, so the
same bits, at every number of K blocks a last trip can have, at every place where a tile's columns meet the next weight scale, and where N ends inside a tile;
and the shapes that take them, on both sides of every line of the rule.  The kernels that ran are checked."""
import pytest
import torch

from oracle import torch_ref as T
from tests import _inputs as I
from tests._routes import kernels

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
    A.require_gpu()
    print("[case]", (M, N, K), pow2, dtype, flush=True)
    quant = T.quant_fp8_e4m3_scale_e8m0 if pow2 else T.quant_block_fp32_scale
    (xq, xs), (wq, ws) = quant(I.act_like(M, K, M + K), (1, 128)), quant(I.weight_like(N, K, N, outliers=False), (128, 128))
    ops = [t.cuda().contiguous() for t in (xq, xs, wq, ws)]
    same_as_columns_apart(M, N, K, ops, pow2, dtype, True)


def same_as_columns_apart(M, N, K, ops, pow2, dtype, wide):
    """The whole product on 128 x 160 tiles (wide) or 128 x 128 ones; column ranges on 128 x 128 ones"""
    from gcore_lowp import _abi as A
    L = A.lib()

    def call(first, last, out):
        w, s = ops[2][first:last], ops[3][first // 128:last // 128]
        A.check(L.lp_gemm_fp8_block(ops[0].data_ptr(), ops[1].data_ptr(), w.data_ptr(), s.data_ptr(), A.E8M0 if pow2 else A.F32, M, last - first, K,
                                    out.data_ptr(), A.BF16 if dtype == torch.bfloat16 else A.F32, None, 0, A.stream_ptr()))

    def product(first, last):
        guard = 4096
        room = torch.full((M * (last - first) + guard,), float("nan"), dtype=dtype, device="cuda")
        call(first, last, room)
        assert bool(room[-guard:].isnan().all())
        return room[:-guard].view(M, last - first)

    ran = kernels(lambda: call(0, N, torch.empty(M, N, dtype=dtype, device="cuda")))
    assert len(ran) == 1 and ("gemm_asmILi128ELi160E" if wide else "gemm_asmILi128ELi128E") in ran[0], ran
    got = product(0, N)
    # column ranges of at most 255 tiles, alike: whole columns of tiles, more than the decode kernels take in slices of 128 rows
    rows, columns = -(-M // 128), N // 128
    parts = -(-columns // max(1, 255 // rows))
    for i in range(parts):
        first, last = (columns * j // parts * 128 for j in (i, i + 1))
        assert not any("ILi160E" in n for n in kernels(lambda: call(first, last, torch.empty(M, last - first, dtype=dtype, device="cuda"))))
        want = product(first, last)
        if not pow2 and K % 1024 == 0:
            # one tile a CU, fp32 scales: two halves of K, added in fp32 at the end; the others add up to 16 K blocks one after the other (6e-8 each of what is there)
            assert ((got[:, first:last].double() - want.double()).norm() / want.double().norm()).item() < 16 * 6e-8
            continue
        bad = (got[:, first:last] != want).nonzero()
        assert not len(bad), (first, last, len(bad), bad[:4].tolist())


# (M, N, K), tiles of 128 x 128, of 128 x 160, whether fp32 and e8m0 scales take the latter
LINES = [
    # two workgroups a CU
    ((1024, 8704, 2176), 544, 440, True, True), ((1000, 8576, 2176), 536, 432, True, False), ((1000, 8704, 1920), 544, 440, True, False),
    ((1024, 8704, 2048), 544, 440, True, True), ((1100, 7808, 2048), 549, 441, True, True),
    ((1200, 7040, 2560), 550, 440, True, True), ((1300, 6400, 2560), 550, 440, True, True), ((1300, 6400, 3072), 550, 440, True, True),
    ((400, 17408, 1024), 544, 436, True, False), ((1000, 8704, 1024), 544, 440, True, False), ((640, 15104, 1024), 590, 475, True, False),
    ((400, 17408, 1152), 544, 436, True, False), ((1000, 8704, 896), 544, 440, False, False), ((1000, 8320, 1152), 520, 416, False, False), ((1000, 8320, 2048), 520, 416, True, False),
    ((1000, 10496, 2176), 656, 528, False, False),                                          # three a CU either way
    # one
    ((1000, 4224, 2048), 264, 216, False, True), ((1000, 4864, 1920), 304, 248, False, True), ((1000, 4224, 1920), 264, 216, False, False),
    ((640, 7680, 1024), 300, 240, False, True), ((640, 7680, 896), 300, 240, False, False), ((512, 9600, 1408), 300, 240, False, True),
    ((1000, 4608, 2816), 288, 232, True, True), ((1000, 4480, 2816), 280, 224, False, True), ((256, 16512, 2816), 258, 208, True, True),
    ((1000, 4864, 2688), 304, 248, True, True), ((640, 7680, 2688), 300, 240, False, True), ((1000, 5120, 2048), 320, 256, True, True), ((300, 13440, 2048), 315, 252, False, True),
    ((1024, 4096, 2944), 256, 208, False, False), ((1000, 5248, 2944), 328, 264, False, False),
]


@pytest.mark.parametrize("pow2", [False, True], ids=["f32scale", "e8m0scale"])
@pytest.mark.parametrize("shape,narrow,wide,with_f32,with_e8m0", LINES, ids=str)
def test_lines_of_the_rule(shape, narrow, wide, with_f32, with_e8m0, pow2):
    from gcore_lowp import _abi as A
    A.require_gpu()
    M, N, K = shape
    assert -(-M // 128) * (N // 128) == narrow and -(-M // 128) * -(-N // 160) == wide
    print("[case]", (M, N, K), pow2, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    xq, wq = (torch.randn(r, K, generator=g, device="cuda").to(torch.float8_e4m3fn) for r in (M, N))
    xs, ws = (torch.randint(120, 126, s, generator=g, device="cuda", dtype=torch.uint8) for s in ((M, K // 128), (N // 128, K // 128)))
    if not pow2:
        xs, ws = (torch.pow(2.0, t.float() - 127) * 1.25 for t in (xs, ws))
    same_as_columns_apart(M, N, K, (xq, xs, wq, ws), pow2, torch.float32, with_e8m0 if pow2 else with_f32)


@pytest.mark.parametrize("knob", ["LP_GEMM_MID_DUAL=0", "LP_GEMM_MID_STAGES=4", "LP_GEMM_MID_KSUB=1"])
def test_knobs_of_the_128_wide_loops_hold(knob):
    """The knobs force a loop of 128 x 128 tiles (they are read once per process, hence the child); a shape that takes 128 x 160 tiles without them."""
    import os
    import subprocess
    import sys
    code = (
        "import torch\n"
        "from gcore_lowp import _abi as A\n"
        "from tests._routes import kernels\n"
        "M, N, K = 1000, 5120, 2560\n"
        "t = [torch.zeros(n, dtype=torch.uint8, device='cuda') for n in (M * K, M * K // 32, N * K, N * K // 4096, 2 * M * N)]\n"
        "print('kernels', *kernels(lambda: A.check(A.lib().lp_gemm_fp8_block(*[x.data_ptr() for x in t[:4]], A.F32, M, N, K, t[4].data_ptr(), A.BF16, None, 0, A.stream_ptr()))))\n")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    print("[case]", knob, flush=True)
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([root] + [p for p in sys.path if p]), **dict([knob.split("=")]))
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, (r.stdout[-1500:], r.stderr[-1500:])
    ran = [line.split()[1:] for line in r.stdout.splitlines() if line.startswith("kernels")]
    assert len(ran) == 1 and len(ran[0]) == 1 and "gemm_asmILi128ELi128E" in ran[0][0], ran
