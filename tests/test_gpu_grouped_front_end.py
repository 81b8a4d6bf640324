"""The grouped linear through the native front end against its wrappers' own way through the C ABI: the same bits, for every form of
the operands, and what the front end does not take goes the wrappers' way."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SPLITS = {
    "ragged": [0, 1, 127, 128, 129, 0, 255, 256, 257, 513, 3, 640],       # every kind of weight-gradient problem, two experts empty
    "one": [130],
    "short": [5, 0, 128, 100],                                            # one K block each
    "long": [1024, 512],                                                  # whole groups of four K blocks
    "513 experts": [int(i % 9 == 0) * 3 for i in range(513)],             # more than a launch's arguments carry
    "many": [int(i % 7 == 0) * 40 for i in range(300)],                   # a table of several thousand bytes
}


@pytest.fixture(scope="module")
def G():
    import gcore_lowp
    return gcore_lowp


def step(G, splits, form, dtype, want_x, want_w, k=256, n=384):
    g = torch.Generator(device="cuda").manual_seed(len(splits) + k)
    rows, E = sum(splits), len(splits)
    x = torch.randn(rows, k, generator=g, device="cuda").to(dtype)
    if form == "three dims":
        x = x.view(1, rows, k)
    elif form == "strided":
        x = torch.cat([x, x], 1)[:, :k]
    elif form == "off 16 bytes":
        x = torch.cat([x.flatten()[:1], x.flatten()])[1:].view(rows, k)
    x = x.detach().requires_grad_(want_x)
    w = (torch.randn(E, n, k, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    layer = G.MyTeGroupedLinearFp8(E)
    if want_w:
        weight = w.requires_grad_(True)
    else:
        q, s = G.quant_fp8_e4m3_scale_e8m0(w.view(E * n, k))
        weight = (q.view(E, n, k), s.view(E, n // 128, k // 128))
    dy = torch.randn(rows, n, generator=g, device="cuda").to(dtype) * 1e-3
    out = layer(x, weight, splits)
    wanted = [t for t, on in ((x, want_x), (w, want_w)) if on]
    grads = torch.autograd.grad(out, wanted, dy.view(out.shape)) if wanted else ()
    return [out.detach(), *grads]


CASES = [(s, "plain", torch.bfloat16, True, True) for s in SPLITS] + [
    ("ragged", f, torch.bfloat16, True, True) for f in ("three dims", "strided", "off 16 bytes")] + [
    ("ragged", "plain", torch.float32, True, True), ("ragged", "plain", torch.bfloat16, False, True), ("ragged", "plain", torch.bfloat16, True, False),
    ("ragged", "plain", torch.bfloat16, False, False), ("ragged", "strided", torch.bfloat16, False, False), ("many", "plain", torch.bfloat16, False, False),
    ("513 experts", "plain", torch.bfloat16, False, False), ("513 experts", "plain", torch.bfloat16, True, False), ("long", "plain", torch.bfloat16, False, False), ("long", "off 16 bytes", torch.bfloat16, True, False)]


@pytest.mark.parametrize("splits,form,dtype,want_x,want_w", CASES, ids=str)
def test_front_end_and_wrappers_give_the_same_bits(G, monkeypatch, splits, form, dtype, want_x, want_w):
    from gcore_lowp import _native
    args = (SPLITS[splits], form, dtype, want_x, want_w)
    print("[case]", splits, form, dtype, want_x, want_w, flush=True)
    taken = []
    for name in ("grouped_forward", "grouped_backward"):
        real = getattr(_native.fast, name)
        monkeypatch.setattr(_native.fast, name, lambda *a, real=real, name=name: [r for r in [real(*a)] if taken.append((name, r is not None)) is None][0])
    got = step(G, *args)
    if form == "plain" and dtype == torch.bfloat16:
        # (the backward leaves more than 512 experts to the wrappers)
        backward = ("grouped_backward", splits != "513 experts")
        assert ("grouped_forward", True) in taken and (not want_x or backward in taken), taken
    for name in ("grouped_forward", "grouped_backward"):
        monkeypatch.setattr(_native.fast, name, lambda *a: None)
    want = step(G, *args)
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("train", [False, True], ids=["inference", "training"])
@pytest.mark.parametrize("splits,k,n,host,device", [
    ([3] * 40, 3328, 1024, "two", "128"), ([3] * 40, 2432, 1024, "128", "128"), ([0, 64, 1] * 30, 1280, 1152, "128", "two"), ([64] * 11 + [65], 1280, 1152, "128", "128"),
    ([1] * 440, 256, 256, "128", "128"), ([1] * 439 + [129] + [0] * 5, 256, 256, "128", "128"), ([0] * 9 + [257, 0, 128], 1152, 640, "128", "128"),
    ([3, 0, 0] * 46, 3456, 1408, "128", "two"), ([200] * 3 + [56] * 9, 2816, 4608, "two", "128")],
    ids=["weights streamed", "K of 19 blocks", "short K", "short K, more rows", "440 row tiles", "441 row tiles", "row tiles of an expert", "a few in a second round", "one round"])
def test_kernel_chosen_by_the_row_counts(G, monkeypatch, splits, k, n, host, device, train):
    """The launch that knows the counts may take tiles of another size than the one that does not: the same sums."""
    from gcore_lowp import _native
    from tests._routes import kernels
    args = (splits, "plain", torch.bfloat16, train, False, k, n)
    names = {"128": "gemm_asm_groupedILi128ELi128E", "two": "gemm_asm_grouped_mixedILb1ELb0E"}      # (the backward's product is grouped_mixed<true, true, ..>)
    print("[case]", len(splits), sum(splits), k, n, train, flush=True)

    def run(wanted):
        layer, x, weight = G.MyTeGroupedLinearFp8(len(splits)), *operands
        forward = [m for m in kernels(lambda: layer(x, weight, splits)) if "gemm_asm_grouped" in m]
        assert len(forward) == 1 and names[wanted] in forward[0], (wanted, forward)
        return step(G, *args)

    g = torch.Generator(device="cuda").manual_seed(5)
    q, s = G.quant_fp8_e4m3_scale_e8m0(torch.randn(len(splits) * n, k, generator=g, device="cuda", dtype=torch.bfloat16))
    operands = (torch.randn(sum(splits), k, generator=g, device="cuda", dtype=torch.bfloat16).requires_grad_(train),
                (q.view(len(splits), n, k), s.view(len(splits), n // 128, k // 128)))
    got = run(host)
    monkeypatch.setattr(_native.fast, "grouped_forward", lambda *a: None)
    want = run(device)
    assert len(got) == len(want) == 1 + train and all(torch.equal(a, b) for a, b in zip(got, want))


def test_front_end_in_a_graph(G):
    """The tables travel in the launches' arguments: a captured layer replays with them."""
    splits = SPLITS["ragged"]
    g = torch.Generator(device="cuda").manual_seed(3)
    E, n, k = len(splits), 384, 256
    x = torch.randn(sum(splits), k, generator=g, device="cuda", dtype=torch.bfloat16)
    q, s = G.quant_fp8_e4m3_scale_e8m0(torch.randn(E * n, k, generator=g, device="cuda", dtype=torch.bfloat16))
    w, layer = (q.view(E, n, k), s.view(E, n // 128, k // 128)), G.MyTeGroupedLinearFp8(E)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.no_grad():
        layer(x, w, splits)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph), torch.no_grad():
        out = layer(x, w, splits)
    for i in range(3):
        x.copy_(torch.randn(x.shape, generator=g, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        with torch.no_grad():
            assert torch.equal(out, layer(x, w, splits)), i


def test_more_experts_than_the_arguments_hold_are_quantised_once(G):
    """The launch that takes the offsets by value refuses; the activations are quantised and the result is allocated once all the same."""
    import ctypes
    from gcore_lowp import _abi as A, _native
    mod, L, calls = _native._load(), A.lib(), []
    restype, argtypes = A.PROTOTYPES["lp_quant_fp8_block"]
    counting = ctypes.CFUNCTYPE(restype, *argtypes)(lambda *a: calls.append(1) or L.lp_quant_fp8_block(*a))
    real = [ctypes.cast(getattr(L, n), ctypes.c_void_p).value for n in _native._BOUND]
    at = _native._BOUND.index("lp_quant_fp8_block")
    splits, (k, n) = SPLITS["513 experts"], (256, 128)
    x = torch.randn(sum(splits), k, device="cuda", dtype=torch.bfloat16)
    q = torch.zeros(len(splits), n, k, device="cuda").to(torch.float8_e4m3fn)
    s = torch.ones(len(splits), n // 128, k // 128, device="cuda").to(torch.float8_e8m0fnu)
    print("[case]", len(splits), "experts", flush=True)
    mod.bind(*real[:at], ctypes.cast(counting, ctypes.c_void_p).value, *real[at + 1:])
    try:
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        out = mod.grouped_forward(x, q, s, splits, A.BF16, False, False)
        made = torch.cuda.memory_stats()["allocation.all.allocated"] - before
    finally:
        mod.bind(*real)
    assert out is not None and len(calls) == 1
    assert made == 4                                     # codes, scales, result, the table with the offsets


def test_row_counts_the_front_end_refuses(G):
    from gcore_lowp import _abi as A, _native
    x = torch.zeros(4, 128, device="cuda", dtype=torch.bfloat16)
    q, s = torch.zeros(2, 128, 128, device="cuda").to(torch.float8_e4m3fn), torch.ones(2, 1, 1, device="cuda").to(torch.float8_e8m0fnu)
    for splits in ([4], [2, 3], [5, -1], (2, 2), [2, 2.0], [1 << 40, 4], [1, 3, 0]):
        assert _native.fast.grouped_forward(x, q, s, splits, A.BF16, False, False) is None, splits
    with pytest.raises(AssertionError):
        G.MyTeGroupedLinearFp8(2)(x, (q, s), [5, -1])
    with pytest.raises(AssertionError):
        G.MyTeGroupedLinearFp8(2)(x, (q, s), [2, 3])
