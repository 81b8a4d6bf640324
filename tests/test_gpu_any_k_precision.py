"""How far the loops that accumulate in the scaled matrix instruction over all K blocks (e8m0 scales) are from the exact product, against
the loops that add each block's partial sum with an fp32 FMA (fp32 scales, here the same powers of two on the same codes): dense, grouped,
on weights stored [K, N] and row-scaled, K from three blocks to 143, fp32 results, float64 product of the codes as the truth.

Both share the instruction's own rounding of a block's 128 products, 1.5e-5 of the result (2-norm) for normal operands of either sign and
2.4e-5 with a few loud channels.  What differs is the rounding of each addition to the running sum, at most 2^-23 of it (the instruction cuts, the FMA rounds to nearest).  For
sums of either sign these are independent: sqrt(143) 2^-23 / 2 = 7e-7 beside 1.5e-5, 0.1 % in quadrature, so 1.01 times.  For sums of one
sign the cuts add up: on average half a unit of a running sum that is on average half the result, B 2^-25 for B blocks (measured: 2.50e-6
-> 2.57e-6 at 143 blocks, 2.50e-6 -> 2.52e-6 at 57, equal up to 8; K in whole groups of four blocks has always been accumulated so)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

E4M3, E8M0 = torch.float8_e4m3fn, torch.float8_e8m0fnu


def deq(q, s, rows):
    return q.double() * s.double().repeat_interleave(128, -1).repeat_interleave(rows, -2)


def error(out, ref):
    return ((out.double() - ref).norm() / ref.norm()).item()


def values(g, rows, cols, one_sign):
    """activations with a few loud channels, or the same without their signs"""
    x = torch.randn(rows, cols, generator=g, device="cuda", dtype=torch.bfloat16)
    x[:, torch.randint(0, cols, (max(1, cols // 512),), generator=g, device="cuda")] *= 10.0
    return x.abs() if one_sign else x


@pytest.mark.parametrize("one_sign", [False, True], ids=["either sign", "one sign"])
@pytest.mark.parametrize("blocks", [3, 7, 23, 57, 143])
@pytest.mark.parametrize("route", ["dense", "grouped", "stored [K, N]", "row-scaled"])
def test_no_further_from_the_product_than_the_folding_loops(route, blocks, one_sign):
    import gcore_lowp as G
    from gcore_lowp import _abi as A
    g = torch.Generator(device="cuda").manual_seed(blocks)
    M, N, K = (1101, 2176, blocks * 128) if route == "dense" else (384, 1152, blocks * 128)      # few dense rows run on kernels without these loops
    xq, xs = G.quant_fp8_e4m3_scale_e8m0(values(g, M, K, one_sign), (1, 128))
    w = values(g, N, K, one_sign) * 0.02
    wq, ws = G.quant_fp8_e4m3_scale_e8m0(w, (1, 128) if route == "row-scaled" else (128, 128))
    ref = deq(xq, xs, 1) @ deq(wq, ws, 1 if route == "row-scaled" else 128).t()
    xf, wf = xs.float(), ws.float()
    f32 = dict(out_dtype=torch.float32)
    if route == "dense":
        scaled = G.gemm_fp8_block_scaling_impl(xq, xs, wq, ws, **f32)
        folded = G.gemm_fp8_block_scaling_impl(xq, xf, wq, wf, **f32)
    elif route == "row-scaled":
        scaled, folded = (torch.empty(M, N, device="cuda") for _ in range(2))
        for out, a_s, b_s, code in ((scaled, xs, ws, A.E8M0), (folded, xf, wf, A.F32)):
            A.check(A.lib().lp_gemm_fp8_rowscale(xq.data_ptr(), a_s.data_ptr(), wq.data_ptr(), b_s.data_ptr(), code, M, N, K,
                                                 out.data_ptr(), A.F32, A.stream_ptr()))
    else:
        offs = torch.tensor([0, 100, M], dtype=torch.int32, device="cuda")         # two experts with the same weights
        wq2, ws2, wf2 = (torch.stack([t.view(torch.uint8) if t.dtype != torch.float32 else t] * 2) for t in (wq, ws, wf))
        folded = G.grouped_gemm_fp8(xq, xf, wq2.view(E4M3), wf2, offs, total_rows=M, **f32)
        if route == "grouped":
            scaled = G.grouped_gemm_fp8(xq, xs, wq2.view(E4M3), ws2.view(E8M0), offs, total_rows=M, **f32)
        else:
            scaled = G.grouped_gemm_fp8_nn(xq, xs, wq2.transpose(1, 2).contiguous().view(E4M3), ws2.transpose(1, 2).contiguous().view(E8M0),
                                           offs, total_rows=M, **f32)
    es, ef = error(scaled, ref), error(folded, ref)
    print("[case]", route, blocks, one_sign, "scaled %.4e folded %.4e" % (es, ef), flush=True)
    assert es <= (ef + blocks * 2.0 ** -25 if one_sign else 1.01 * ef)
