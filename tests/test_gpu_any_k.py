"""The GEMM loops that take any number of K blocks (K a multiple of 128 and not of 512), at their edges: one block up to two
trips of four and a remainder of each length, row and column tiles that end inside the problem, both scale types, the dense
kernels of both tile sizes, the grouped kernels of all three and the one on weights stored [K, N].  Against fp32
dequantise-then-matmul: the bf16 result is off by at most half a unit in its last place, 2^-8 of a value just above a power of
two, plus what the matrix instruction drops of a block's 128 products, measured as at most 3.9e-5 of the largest result, which
is at most 6.3 times the results' root mean square here: 2.5e-4 of that.  So the error is at most 2^-8 + 2^-12 of the larger of
the element and the root mean square."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = 2.0 ** -8 + 2.0 ** -12


@pytest.fixture(scope="module")
def G():
    import gcore_lowp
    return gcore_lowp


def deq(q, s, rows):
    return q.float() * s.float().repeat_interleave(128, -1).repeat_interleave(rows, -2)


def close(out, ref, what):
    out, rms = out.float(), ref.square().mean().sqrt().clamp(min=1e-30)
    err = ((out - ref).abs() / ref.abs().clamp(min=rms)).max().item()
    print("[case]", what, "%.2e" % err, flush=True)
    assert torch.isfinite(out).all() and err <= BOUND, (what, err)


def operands(G, M, N, K, pow2, seed, experts=None):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16)
    w = torch.randn((experts or 1) * N, K, generator=g, device="cuda", dtype=torch.bfloat16) * 0.02
    if pow2:
        (xq, xs), (wq, ws) = G.quant_fp8_e4m3_scale_e8m0(x, (1, 128)), G.quant_fp8_e4m3_scale_e8m0(w)
    else:
        (xq, xs), (wq, ws) = G.quant_1d(x), G.quant_2d(w)
    if experts is not None:
        wq, ws = wq.view(experts, N, K), ws.view(experts, N // 128, K // 128)
    return xq, xs, wq, ws


@pytest.mark.parametrize("pow2", [False, True], ids=["f32scale", "e8m0scale"])
@pytest.mark.parametrize("blocks", [1, 2, 3, 5, 6, 7, 9, 23])
@pytest.mark.parametrize("M,N", [(1101, 2176), (3401, 4224)], ids=["tiles128", "tiles256"])
def test_dense(G, M, N, blocks, pow2):
    K = blocks * 128
    xq, xs, wq, ws = operands(G, M, N, K, pow2, blocks)
    out = G.gemm_fp8_block_scaling_impl(xq, xs, wq, ws)
    close(out, deq(xq, xs, 1) @ deq(wq, ws, 128).t(), ("dense", M, N, K, pow2))


@pytest.mark.parametrize("pow2", [False, True], ids=["f32scale", "e8m0scale"])
@pytest.mark.parametrize("splits,N,K", [([700, 0, 3, 257, 128, 129, 1, 64] * 4, 2176, 384), ([1000, 1, 0, 260, 385, 60] * 6, 1152, 1408),
                                        ([33, 0, 300, 1], 640, 640), ([5, 2, 0, 129, 64], 384, 1152), ([600, 0, 60, 1] * 20, 896, 1024), ([1100, 1283], 640, 512), ([2945], 384, 1024)],
                         ids=lambda v: str(v) if isinstance(v, int) else "E%d" % len(v))
def test_grouped(G, splits, N, K, pow2):
    E, M = len(splits), sum(splits)
    xq, xs, wq, ws = operands(G, M, N, K, pow2, N + K, E)
    offs = torch.tensor([0] + torch.tensor(splits).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    out = G.grouped_gemm_fp8(xq, xs, wq, ws, offs, total_rows=M)
    xd = deq(xq, xs, 1)
    ref = torch.cat([xd[offs[e]:offs[e + 1]] @ deq(wq[e], ws[e], 128).t() for e in range(E)])
    close(out, ref, ("grouped", E, M, N, K, pow2))


@pytest.mark.parametrize("splits,N,K", [([700, 0, 3, 257, 128, 129, 1, 64], 640, 384), ([300, 0, 60], 1408, 1152), ([1, 500], 128, 128),
                                        ([64, 0, 200], 2304, 640), ([40, 300], 1024, 896)],
                         ids=lambda v: str(v) if isinstance(v, int) else "E%d" % len(v))
def test_grouped_nn(G, splits, N, K):
    E, M = len(splits), sum(splits)
    xq, xs, _, _ = operands(G, M, N, K, True, N + K, E)
    wq, ws = G.quant_fp8_e4m3_scale_e8m0((torch.randn(E * K, N, device="cuda") * 0.05).to(torch.bfloat16))
    wq, ws = wq.view(E, K, N), ws.view(E, K // 128, N // 128)
    offs = torch.tensor([0] + torch.tensor(splits).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    out = G.grouped_gemm_fp8_nn(xq, xs, wq, ws, offs, total_rows=M)
    xd = deq(xq, xs, 1)
    ref = torch.cat([xd[offs[e]:offs[e + 1]] @ deq(wq[e], ws[e], 128) for e in range(E)])
    close(out, ref, ("grouped nn", E, M, N, K))
