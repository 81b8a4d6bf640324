"""Dense products cut along K (partial sums of ranges of K blocks in fp32, added by a second launch) against the same call without
scratch, which takes every tile whole."""
import pytest
import torch

from oracle import torch_ref as T
from tests import _inputs as I

pytestmark = pytest.mark.gpu

CASES = [
    (65, 1152, 12544),      # nine tiles, one row of the second half; ranges shorter than a trip of four K blocks
    (70, 7680, 10368),      # one row of tiles
    (129, 128, 7168),       # two tiles, the second of one row
    (200, 256, 5120),
    (257, 2176, 12416),     # 97 K blocks: the last range shorter
    (512, 512, 7168),       # K % 512 == 0: aligned loop
    (640, 1920, 11392),
    (1000, 4992, 6016),     # 312 tiles: 32 columns of them whole, seven cut
    (1537, 2688, 9344),     # the last row tile of one row
    (64, 5120, 6144), (56, 4224, 7168), (33, 5120, 7296), (24, 5120, 8192), (17, 5376, 14464), (70, 4096, 7168),      # ahead of the decode kernels
    (47, 2432, 15232),      # up to 64 rows without a decode kernel for this K
]


def _call(L, A, ops, sdt, M, N, K, dtype, scratch, cut=None):
    """`cut`: whether the call must have written partial sums to its scratch"""
    out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    ws = torch.full((max(scratch, 16) // 4,), float("nan"), device="cuda")
    A.check(L.lp_gemm_fp8_block(*(t.data_ptr() for t in ops), sdt, M, N, K, out.data_ptr(), A.BF16 if dtype == torch.bfloat16 else A.F32,
                                ws.data_ptr() if scratch else None, scratch, A.stream_ptr()))
    assert cut is None or bool((~ws.isnan()).any()) == cut
    return out


@pytest.mark.parametrize("pow2", [False, True], ids=["f32scale", "e8m0scale"])
@pytest.mark.parametrize("M,N,K", CASES, ids=str)
def test_ranges_against_whole_tiles(M, N, K, pow2):
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    need = L.lp_gemm_split_workspace_bytes(M, N, K)
    print("[case]", (M, N, K), "e8m0" if pow2 else "f32", need, flush=True)
    assert 0 < need <= 20 << 20
    # with e8m0 scales the decode kernels keep their shapes, whatever the scratch
    cuts = not pow2 or L.lp_gemm_block_workspace_bytes(A.E8M0, M, N, K) > 0
    assert cuts or M <= 128
    x, w = I.act_like(M, K, M + K), I.weight_like(N, K, N, outliers=False)
    quant = T.quant_fp8_e4m3_scale_e8m0 if pow2 else T.quant_block_fp32_scale
    (xq, xs), (wq, ws) = quant(x, (1, 128)), quant(w, (128, 128))
    ops = [t.cuda().contiguous() for t in (xq, xs, wq, ws)]
    sdt = A.E8M0 if pow2 else A.F32
    exact = torch.zeros(M, N, dtype=torch.float64, device="cuda")
    for k in range(0, K, 128):
        b = slice(k, k + 128)
        part = ops[0][:, b].double() @ ops[2][:, b].double().t()
        exact += part * ops[1][:, k // 128].double()[:, None] * ops[3][:, k // 128].double().repeat_interleave(128)[None, :]
    whole, cut = (_call(L, A, ops, sdt, M, N, K, torch.float32, n, n > 0 and cuts) for n in (0, need))
    assert cuts or torch.equal(whole, cut)
    err = [((o.double() - exact).norm() / exact.norm()).item() for o in (whole, cut)]
    # the matrix instruction's own error, 1.5e-5 over one K block and over many (up to 2.5e-5 with loud channels); up to 16 ranges are
    # added in fp32 (half an ulp, 6e-8 each: 3e-4 of that error)
    assert err[1] <= max(err[0], 1e-6) * 1.002 and err[1] < 4e-5, err
    narrow = _call(L, A, ops, sdt, M, N, K, torch.bfloat16, need, cuts)
    assert torch.equal(narrow, cut.to(torch.bfloat16))                   # the same sums, rounded once
    assert torch.equal(cut, _call(L, A, ops, sdt, M, N, K, torch.float32, need))
    # less scratch than the plan's: fewer ranges or none, same result within the same error
    for n in (need // 2, need // 16 & ~15):
        less = _call(L, A, ops, sdt, M, N, K, torch.float32, n)
        assert ((less.double() - exact).norm() / exact.norm()).item() <= max(err[0], 1e-6) * 1.002


@pytest.mark.parametrize("M,N,K", [(100, 2048, 16384), (64, 1024, 18432), (65, 1152, 12544), (129, 128, 7168), (512, 512, 7168), (200, 256, 5120), (927, 128, 4096)], ids=str)
def test_e8m0_ranges_of_few_tiles_fold_every_block(M, N, K):
    """Power-of-two scales as fp32 take the same plan, fold every K block by an fp32 FMA and scale exactly: the same bits.  Operands of one sign,
    on which sums left to the matrix instruction differ by up to 0.2 % of the error."""
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    print("[case]", (M, N, K), flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + K)
    xq, wq = (torch.randn(r, K, generator=g, device="cuda").abs().mul_(8).to(torch.float8_e4m3fn) for r in (M, N))
    xs, ws = (torch.randint(120, 126, s, generator=g, device="cuda", dtype=torch.uint8) for s in ((M, K // 128), (N // 128, K // 128)))
    f32 = [torch.pow(2.0, t.float() - 127) for t in (xs, ws)]
    need = L.lp_gemm_split_workspace_bytes(M, N, K)
    folded = _call(L, A, (xq, f32[0], wq, f32[1]), A.F32, M, N, K, torch.float32, need, True)
    assert torch.equal(_call(L, A, (xq, xs, wq, ws), A.E8M0, M, N, K, torch.float32, need, True), folded)


@pytest.mark.parametrize("M,N,K", [(384, 512, 7168), (65, 1152, 7168), (4000, 128, 7168), (1000, 512, 4608), (33, 5120, 7296)], ids=str)
def test_workspace_of_the_promised_size_and_the_built_in_buffer_agree(M, N, K):
    """lp_gemm_fp8_block with lp_gemm_workspace_bytes and lp_gemm_fp8_block_static: the same plan, whatever room the former has for scale copies."""
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    print("[case]", (M, N, K), flush=True)
    (xq, xs), (wq, ws) = (T.quant_block_fp32_scale(t, b) for t, b in ((I.act_like(M, K, 1), (1, 128)), (I.weight_like(N, K, 2, outliers=False), (128, 128))))
    ops = [t.cuda().contiguous() for t in (xq, xs, wq, ws)]
    want = _call(L, A, ops, A.F32, M, N, K, torch.float32, L.lp_gemm_workspace_bytes(M, N, K))
    got = torch.full((M, N), float("nan"), device="cuda")
    A.check(L.lp_gemm_fp8_block_static(*(t.data_ptr() for t in ops), A.F32, M, N, K, got.data_ptr(), A.F32, A.stream_ptr()))
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K", [(65, 128, 12544), (129, 128, 7168), (65, 1152, 12544), (200, 256, 5120), (1041, 128, 16384), (100, 3072, 9216), (700, 128, 4736)], ids=str)
def test_promised_workspace_holds_the_best_plan(M, N, K):
    """Few tiles: partial sums need no room for rows beyond M, so lp_gemm_workspace_bytes holds as many ranges as a larger workspace, with whole tiles of rows, is used for."""
    from gcore_lowp import _abi as A
    L = A.lib()
    A.require_gpu()
    print("[case]", (M, N, K), flush=True)
    (xq, xs), (wq, ws) = (T.quant_block_fp32_scale(t, b) for t, b in ((I.act_like(M, K, 1), (1, 128)), (I.weight_like(N, K, 2, outliers=False), (128, 128))))
    ops = [t.cuda().contiguous() for t in (xq, xs, wq, ws)]
    promised, best = L.lp_gemm_workspace_bytes(M, N, K), L.lp_gemm_split_workspace_bytes(M, N, K)
    assert promised > 0 and best > 0
    got = _call(L, A, ops, A.F32, M, N, K, torch.float32, promised)
    assert torch.equal(got, _call(L, A, ops, A.F32, M, N, K, torch.float32, best))
    assert not torch.equal(got, _call(L, A, ops, A.F32, M, N, K, torch.float32, 0))            # it is cut at all


def test_ranges_in_a_graph():
    """Captured with its scratch and replayed: every replay is the eager call's result."""
    import gcore_lowp as G
    g = torch.Generator(device="cuda").manual_seed(5)
    M, N, K = 145, 2176, 7424
    xq, xs = G.quant_1d(torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16))
    wq, ws = G.quant_2d(torch.randn(N, K, generator=g, device="cuda", dtype=torch.bfloat16) * 0.02)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        G.gemm_fp8_block_scaling_impl(xq, xs, wq, ws)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = G.gemm_fp8_block_scaling_impl(xq, xs, wq, ws)
    for i in range(3):
        q, s = G.quant_1d(torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16))
        xq.copy_(q)
        xs.copy_(s)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, G.gemm_fp8_block_scaling_impl(xq, xs, wq, ws)), i


@pytest.mark.parametrize("native", [True, False])
def test_decode_kernels_get_no_scratch(monkeypatch, native):
    """e8m0 scales at shapes whose fp32 form is cut: the call allocates its result and nothing else."""
    import gcore_lowp as G
    from gcore_lowp import mygemm_fp8
    if not native:
        class Nothing:
            gemm = staticmethod(lambda *a: None)
        monkeypatch.setattr(mygemm_fp8, "fast", Nothing)
    M, N, K = 48, 8192, 9216
    xq, xs = G.quant_fp8_e4m3_scale_e8m0(torch.ones(M, K, device="cuda", dtype=torch.bfloat16), (1, 128))
    wq, ws = G.quant_fp8_e4m3_scale_e8m0(torch.ones(N, K, device="cuda", dtype=torch.bfloat16))
    print("[case]", (M, N, K), native, flush=True)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = G.gemm_fp8_block_scaling_impl(xq, xs, wq, ws)
    assert torch.cuda.max_memory_allocated() - before == out.numel() * 2


@pytest.mark.parametrize("native", [True, False])
def test_no_room_for_scratch_is_no_error(monkeypatch, native):
    """Memory for the result and not for the partial sums: the call runs as one without scratch does."""
    import gcore_lowp as G
    from gcore_lowp import _abi as A, mygemm_fp8
    if not native:
        class Nothing:
            gemm = staticmethod(lambda *a: None)
        monkeypatch.setattr(mygemm_fp8, "fast", Nothing)
    L, (M, N, K) = A.lib(), (96, 5120, 14720)
    g = torch.Generator(device="cuda").manual_seed(9)
    xq, xs = G.quant_1d(torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16))
    wq, ws = G.quant_2d(torch.randn(N, K, generator=g, device="cuda", dtype=torch.bfloat16))
    want = _call(L, A, (xq, xs, wq, ws), A.F32, M, N, K, torch.bfloat16, 0)
    need = L.lp_gemm_split_workspace_bytes(M, N, K)
    print("[case]", (M, N, K), native, flush=True)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    taken = []
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (6 << 20)) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):          # what the cached segments still have room for goes first
            while True:
                taken.append(torch.empty(need, dtype=torch.uint8, device="cuda"))
        got = G.gemm_fp8_block_scaling_impl(xq, xs, wq, ws)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want)
