"""The native front end of the calls made most often (csrc/host/native.cpp): its answers are those of the wrappers' own way
through the C ABI, what goes wrong in it reaches Python as it does there, and other threads run meanwhile."""
import contextlib
import ctypes
import subprocess
import threading
import time

import pytest
import torch

pytestmark = pytest.mark.gpu

E4M3, E8M0 = torch.float8_e4m3fn, torch.float8_e8m0fnu


@pytest.fixture(scope="module")
def G():
    import gcore_lowp
    return gcore_lowp


def calls(G, rows=256, cols=1024):
    """name -> a call of a public function on operands the front end takes"""
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g, device="cuda", dtype=torch.bfloat16)
    q, s = G.quant_fp8_e4m3_scale_e8m0(x)
    packed = torch.randint(-128, 128, (rows, cols // 2), generator=g, device="cuda", dtype=torch.int8)
    fs = torch.randint(117, 128, (rows, cols // 32), generator=g, device="cuda", dtype=torch.uint8).view(E8M0)
    aq, sa = G.quant_1d(x)
    bq, sb = G.quant_2d(x)
    return {
        "quant_1d": lambda: G.quant_1d(x),
        "quant_1d_pow2": lambda: G.quant_1d(x, round_sf=True),
        "quant_e8m0": lambda: G.quant_fp8_e4m3_scale_e8m0(x),
        "dequant_fp8": lambda: G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(q, s),
        "dequant_fp4": lambda: G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(packed, fs),
        "fp4_rebase": lambda: G.cast_e2m1fn_to_e4m3fn(packed, fs),
        "fp4_rebase_f32": lambda: G.official_expert_to_sgl(packed, fs),
        "fp4_amax": lambda: G.fp4_to_fp8_blockwise(packed, fs),
        "gemm": lambda: G.gemm_fp8_block_scaling_impl(aq, sa, bq, sb),
        "gemm_f32": lambda: G.gemm_fp8_block_scaling_impl(aq, sa, bq, sb, out_dtype=torch.float32),
    }


NAMES = ["quant_1d", "quant_1d_pow2", "quant_e8m0", "dequant_fp8", "dequant_fp4", "fp4_rebase", "fp4_rebase_f32", "fp4_amax", "gemm", "gemm_f32"]


def parts(r):
    return list(r) if isinstance(r, tuple) else [r]


def bits(t):
    return t.contiguous().view(torch.uint8)


@contextlib.contextmanager
def no_more_memory():
    """The allocator has nothing of 16 MB left (a limit of its own: the card is not filled; what it has cached is taken)."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    taken = []
    try:
        with contextlib.suppress(torch.OutOfMemoryError):
            while len(taken) < 1024:
                taken.append(torch.empty(16 << 20, dtype=torch.uint8, device="cuda"))
        yield
    finally:
        taken.clear()
        torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.parametrize("name", NAMES)
def test_out_of_memory_is_torchs_own_error(G, name):
    """A caller that catches torch.OutOfMemoryError, frees and tries again."""
    call = calls(G, 8192, 8192)[name]
    print("[case]", name, flush=True)
    want = [bits(t).clone() for t in parts(call())]
    with no_more_memory():
        with pytest.raises(torch.OutOfMemoryError):
            call()
    got = parts(call())
    assert all(torch.equal(bits(a), b) for a, b in zip(got, want))


# What the front end calls instead of the library: waits (two seconds at most) until another thread says go, and refuses.
STAND_IN = """
#include <unistd.h>
volatile int inside, go, late;
int failed_launch(void) { return %d; }
int stand_in(void) { inside = 1; for (int i = 0; i < 2000; ++i) { if (go) return -1; usleep(1000); } late = 1; return -1; }
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    d = tmp_path_factory.mktemp("stand_in")
    (d / "s.c").write_text(STAND_IN % -3)
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "s.so"), str(d / "s.c")])
    return ctypes.CDLL(str(d / "s.so"))


HOST_ONLY = {"lp_gemm_block_workspace_bytes", "lp_host_flag"}          # answer on the host, without a launch


@contextlib.contextmanager
def bound(function):
    """The front end's module with `function` in the place of the library's entries that launch."""
    from gcore_lowp import _abi as A, _native
    mod = _native._load()
    assert HOST_ONLY <= set(_native._BOUND)
    real = [ctypes.cast(getattr(A.lib(), n), ctypes.c_void_p).value for n in _native._BOUND]
    fake = ctypes.cast(function, ctypes.c_void_p).value
    mod.bind(*[a if n in HOST_ONLY else fake for n, a in zip(_native._BOUND, real)])
    try:
        yield mod
    finally:
        mod.bind(*real)


@pytest.mark.parametrize("name", ["quant_fp8", "quant_fp8_checked", "dequant", "fp4_to_fp8", "gemm", "grouped_forward", "grouped_backward"])
def test_other_threads_run_while_a_launch_waits(G, stand_in, name):
    """A launch can wait for room in a full queue, an allocation for the device."""
    from gcore_lowp import _abi as A
    x = torch.zeros(128, 256, device="cuda", dtype=torch.bfloat16)
    (q, s), packed = G.quant_2d(x), torch.zeros(128, 128, device="cuda", dtype=torch.int8)
    fs, (aq, sa) = torch.ones(128, 8, device="cuda").to(E8M0), G.quant_1d(x)
    experts = q.view(1, 128, 256), torch.ones(1, 1, 2, device="cuda").to(E8M0)
    offsets = torch.tensor([0, 128], device="cuda", dtype=torch.int32)
    word = {n: ctypes.c_int.in_dll(stand_in, n) for n in ("inside", "go", "late")}
    for w in word.values():
        w.value = 0

    def other():
        while not word["inside"].value and not word["late"].value:
            time.sleep(0.001)
        word["go"].value = 1

    with bound(stand_in.stand_in) as mod:
        call = {"quant_fp8": lambda: mod.quant_fp8(x, 1, 128, A.SCALE_DIV, A.F32, A.ZERO_NONE, 1e-12, False),
                "quant_fp8_checked": lambda: mod.quant_fp8(x, 128, 128, A.SCALE_POW2, A.E8M0, A.ZERO_NONE, 0.0, True),
                "dequant": lambda: mod.dequant(q, s, False, A.FP4_NEG_ZERO, A.BF16),
                "fp4_to_fp8": lambda: mod.fp4_to_fp8(packed, fs, 1, A.SCALE_DIV, A.ZERO_NONE, A.F32, 1e-12),
                "gemm": lambda: mod.gemm(aq, sa, q, s, A.BF16),
                "grouped_forward": lambda: mod.grouped_forward(x, *experts, [128], A.BF16, False, False),
                "grouped_backward": lambda: mod.grouped_backward(x[:, :128].contiguous(), *(t.view(torch.uint8) for t in experts), offsets, None, None, None,
                                                                 [128], True, False, A.BF16)}[name]
        t = threading.Thread(target=other)
        t.start()
        r = call()
        t.join()
    assert word["inside"].value == 1 and r is None
    assert not word["late"].value, "no other thread ran during the call"


def test_counter_outlives_a_launch_that_reports_an_error(G, stand_in):
    """The runtime's last error may be an earlier call's, the quantiser queued all the same and the NaN counter in pinned memory
    still to be written: the call ends behind everything queued, and the counter's memory is given back only then."""
    from gcore_lowp import _abi as A
    x = torch.zeros(128, 128, device="cuda", dtype=torch.bfloat16)
    with bound(stand_in.failed_launch) as mod:
        torch.cuda._sleep(20_000_000)
        assert mod.quant_fp8(x, 128, 128, A.SCALE_POW2, A.E8M0, A.ZERO_NONE, 0.0, True) is None
        assert torch.cuda.current_stream().query()


class Counted:
    """Counts what the front end answered and what it left to the wrapper."""

    def __init__(self, monkeypatch):
        from gcore_lowp import _native
        mod = _native._load()
        self.answered, self.left = 0, 0
        for n in _native._ENTRIES:
            monkeypatch.setattr(_native.fast, n, self.counting(getattr(mod, n)), raising=False)

    def counting(self, f):
        def entry(*args):
            r = f(*args)
            if r is None:
                self.left += 1
            else:
                self.answered += 1
            return r
        return entry


@pytest.fixture
def counted(monkeypatch):
    return Counted(monkeypatch)


@contextlib.contextmanager
def without_front_end(monkeypatch):
    from gcore_lowp import _native
    with monkeypatch.context() as m:
        for n in _native._ENTRIES:
            m.setattr(_native.fast, n, lambda *args: None, raising=False)
        yield


def same(a, b):
    return all(x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride() and x.device == y.device
               and torch.equal(bits(x), bits(y)) for x, y in zip(parts(a), parts(b))) and len(parts(a)) == len(parts(b))


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("rows,cols", [(128, 128), (256, 1024), (1152, 640)])
def test_answers_are_the_wrappers(G, counted, monkeypatch, name, rows, cols):
    call = calls(G, rows, cols)[name]
    before = counted.answered
    got = call()
    assert counted.answered == before + 1 and not counted.left, "the front end takes this call"
    with without_front_end(monkeypatch):
        want = call()
    assert same(got, want)


def views(t):
    """the values of t in other clothes: a stride in rows, in columns, an offset that is not aligned"""
    wide = torch.zeros(t.shape[0], t.shape[1] * 2, dtype=t.dtype, device=t.device)
    wide[:, :t.shape[1]].copy_(t)
    apart = torch.zeros(t.shape[1], t.shape[0], dtype=t.dtype, device=t.device)
    apart.copy_(t.t())
    shifted = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    shifted.copy_(t)
    return {"rows apart": wide[:, :t.shape[1]], "transposed": apart.t(), "shifted": shifted}


@pytest.mark.parametrize("clothes", ["rows apart", "transposed", "shifted", "on the host", "half", "leading dims"])
def test_what_is_not_plain_is_answered_as_before(G, monkeypatch, counted, clothes):
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(256, 384, generator=g, device="cuda", dtype=torch.bfloat16)
    if clothes == "on the host":
        y = x.cpu()
    elif clothes == "half":
        y = x.half()
    elif clothes == "leading dims":
        y = x.view(2, 128, 384)
    else:
        y = views(x)[clothes]
    for f in (G.quant_1d, G.quant_fp8_e4m3_scale_e8m0, lambda t: G.quant_fp8_e4m3_scale_e8m0(t, (1, 128)), lambda t: G.quant_1d(t, 32)):
        got = f(y)
        with without_front_end(monkeypatch):
            want = f(y)
        assert same(got, want), clothes
    if clothes in ("rows apart", "transposed", "on the host", "half"):
        assert not counted.answered
    if clothes in ("rows apart", "transposed"):
        q, s = G.quant_fp8_e4m3_scale_e8m0(x)
        v = views(q.view(torch.uint8))[clothes].view(E4M3) if clothes == "rows apart" else q.t().contiguous().t()
        before = counted.answered
        assert same(G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(v, s), G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(q, s))
        assert counted.answered == before + 1                      # the plain one alone


def test_refusals_are_the_wrappers(G, counted):
    x = torch.zeros(128, 256, device="cuda", dtype=torch.bfloat16)
    q, s = G.quant_fp8_e4m3_scale_e8m0(x)
    aq, sa = G.quant_1d(x)
    bq, sb = G.quant_2d(x)
    counted.answered = 0
    with pytest.raises(ValueError, match="not divisible"):
        G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(q, s.view(torch.uint8).repeat(3, 1).view(E8M0))
    with pytest.raises(ValueError, match="leading dims"):
        G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(q.view(torch.uint8).expand(2, 128, 256).contiguous().view(E4M3),
                                                 s.view(torch.uint8).expand(3, 1, 2).contiguous().view(E8M0))
    with pytest.raises(AssertionError):
        G.quant_fp8_e4m3_scale_e8m0(x[:100])
    with pytest.raises(AssertionError):
        G.gemm_fp8_block_scaling_impl(aq, sa[:64], bq, sb)
    with pytest.raises(AssertionError):
        G.gemm_fp8_block_scaling_impl(aq, sa, bq, sb, out_dtype=torch.float16)
    with pytest.raises(AssertionError):
        G.cast_e2m1fn_to_e4m3fn(torch.zeros(100, 64, device="cuda", dtype=torch.int8), torch.ones(100, 4, device="cuda").to(E8M0))
    for empty in (x[:0], x[:, :0]):
        with contextlib.suppress(Exception):
            G.quant_1d(empty)
    assert not counted.answered


@pytest.mark.parametrize("bad", [None, 0, 1000, 16383])
@pytest.mark.parametrize("queue", ["empty", "long"])
def test_nan_check_on_a_stream_of_its_own(G, counted, bad, queue):
    """The flag is waited for on the stream the call was made on, for longer than it is watched (200 us) where much is queued in
    front of it; every call has a counter of its own."""
    side = torch.cuda.Stream()
    x = torch.randn(128, 16384, device="cuda", dtype=torch.bfloat16)
    if bad is not None:
        x[7, bad] = float("nan")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(3):
            if queue == "long":
                torch.cuda._sleep(20_000_000)
            queued = torch.cuda.Event()
            queued.record()
            if bad is None:
                q, s = G.quant_fp8_e4m3_scale_e8m0(x)
                assert queued.query(), "the answer is that of everything queued before"
            else:
                with pytest.raises(AssertionError, match="contains NaN"):
                    G.quant_fp8_e4m3_scale_e8m0(x)
    assert counted.answered == 3
    if bad is None:
        torch.cuda.synchronize()
        want = G.quant_fp8_e4m3_scale_e8m0(x)
        assert same((q, s), want)


def test_every_block_with_a_nan_is_seen(G):
    x = torch.zeros(1024, 2048, device="cuda", dtype=torch.bfloat16)
    for r in range(0, 1024, 128):
        for c in range(0, 2048, 128):
            x.zero_()
            x[r + 77, c + 11] = float("nan")
            with pytest.raises(AssertionError, match="contains NaN"):
                G.quant_fp8_e4m3_scale_e8m0(x)


@pytest.mark.parametrize("name", [n for n in NAMES if n != "quant_e8m0"])
def test_captured_calls(G, counted, name):
    """Under capture the front end answers too; replays, with other work between them, give the eager result each time."""
    call = calls(G)[name]
    want = [bits(t).clone() for t in parts(call())]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    before = counted.answered
    with torch.cuda.graph(graph):
        got = parts(call())
    assert counted.answered == before + 1
    for _ in range(3):
        for t in got:
            bits(t).zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(bits(a), b) for a, b in zip(got, want)), name
        call()


def test_threads_with_streams_of_their_own(G):
    """Calls from several threads at once, each on its own stream and its own operands."""
    wrong = []

    def work(seed):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                g = torch.Generator(device="cuda").manual_seed(seed)
                x = torch.randn(256, 512 + 128 * seed, generator=g, device="cuda", dtype=torch.bfloat16)
                first = None
                for _ in range(20):
                    q, s = G.quant_fp8_e4m3_scale_e8m0(x)
                    aq, sa = G.quant_1d(x)
                    c = G.gemm_fp8_block_scaling_impl(aq, sa, *G.quant_2d(x))
                    back = G.dequant_fp4_e2m1_fp8_scale_e8m0_packed(q, s)
                    r = [bits(t).clone() for t in (q, s, aq, sa, c, back)]
                    first = first or r
                    if not all(torch.equal(a, b) for a, b in zip(r, first)):
                        wrong.append((seed, "differs from its first result"))
                assert (back.float() - x.float()).abs().max() <= x.float().abs().max() / 16
        except BaseException as e:
            wrong.append((seed, repr(e)))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong, wrong
