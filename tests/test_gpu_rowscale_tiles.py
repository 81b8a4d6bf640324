"""The row-scaled grouped GEMM on both tile sizes of its loop: matrices that end inside a tile, in rows (where half of the waves
have no row of their own and still stage the scales of the tile's columns), in columns and in both, three K blocks up to two trips
of four and each remainder, an unaligned scale table (an odd number of blocks in front), and the loop for K in whole groups of four
blocks.  Bound as in tests/test_gpu_any_k.py."""
import pytest
import torch

from tests.test_gpu_any_k import close, deq

pytestmark = pytest.mark.gpu


def tile_rows(M, N, looped, kb):
    """launch_rowscale_asm of csrc/gemm_fp8_big.hip, for a list of `looped` problems of up to kb blocks"""
    big, small = -(-M // 256) * -(-N // 256) * looped, -(-M // 128) * -(-N // 128) * looped
    rounds = -(-big // 256)
    cost = (83 if kb >= 32 else 88 if kb >= 16 else 90 if kb >= 11 else 92 if kb >= 8 else 92 + 4 // rounds if kb >= 5
            else 98 + 10 // rounds if looped == 1 else 94 + 8 // rounds)
    paid = rounds * cost if looped == 1 else big * cost // 256 + 10
    return 256 if big >= 256 and paid < small * 100 // 1024 + 8 else 128


@pytest.mark.parametrize("M,N,tile", [(384, 640, 128), (1408, 2048, 128), (2304, 4096, 256), (2048, 2176, 256), (2176, 2048, 256), (1408, 4096, 256),
                                      (2688, 2688, 256), (1920, 3968, 256)],
                         ids=["tiles128", "tiles128_1408", "tiles256", "tiles256_ragged_columns", "tiles256_ragged_rows", "tiles256_ragged_rows_1408",
                              "tiles256_ragged_both", "tiles256_ragged_both_1920"])
def test_problems_of_any_length(M, N, tile):
    import gcore_lowp as G
    k_blocks = [3, 9, 1, 4, 5, 2, 8, 6, 7, 0, 11]
    assert tile_rows(M, N, sum(kb > 2 for kb in k_blocks), 11) == tile
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


@pytest.mark.parametrize("E,M,N", [(1, 128, 128), (3, 384, 640), (4, 1408, 1024), (9, 2048, 2176), (3, 4096, 4096)])
def test_whole_groups_of_four_blocks(E, M, N):
    """Problems whose K blocks are all multiples of four, with and without one beside them that has three: the loops for such K and
    for any agree in every bit, on their own tile size or another; one problem by itself too."""
    import gcore_lowp as G
    k_blocks = [4 * (1 + e % 3) for e in range(E)]
    g = torch.Generator(device="cuda").manual_seed(E)
    ops = [G.quant_fp8_e4m3_scale_e8m0(torch.randn(M, kb * 128, generator=g, device="cuda", dtype=torch.bfloat16), (1, 128))
           + G.quant_fp8_e4m3_scale_e8m0(torch.randn(N, kb * 128, generator=g, device="cuda", dtype=torch.bfloat16) * 0.05, (1, 128))
           for kb in k_blocks + [3]]
    flat = [[o[i].view(torch.uint8).flatten() for o in ops] for i in range(4)]
    print("[case]", E, M, N, flush=True)
    out = torch.full((E, M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    G.gemm_fp8_rowscale_grouped(*(torch.cat(f[:E]) for f in flat), k_blocks, M, N, out)
    for e, o in enumerate(ops[:E]):
        close(out[e], deq(o[0], o[1], 1) @ deq(o[2], o[3], 1).t(), ("whole groups", M, N, k_blocks[e]))
    both = torch.full((E + 1, M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    G.gemm_fp8_rowscale_grouped(*(torch.cat(f) for f in flat), k_blocks + [3], M, N, both)
    assert torch.equal(both[:E], out)
    one = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    G.gemm_fp8_rowscale(*(f[E - 1] for f in flat), M, N, k_blocks[-1] * 128, one)
    assert torch.equal(one, out[E - 1])


@pytest.mark.parametrize("k_in,tile", [(1152, 128), (2048, 256), (3840, 256)])
def test_weight_gradient_of_a_layer_whose_width_ends_inside_a_tile(k_in, tile):
    """The grouped linear's dW, 1408 = 5.5 x 256 output features, experts of 513 .. 1400 rows (5 to 11 K blocks): expert by expert
    against the product of the same quantised operands in fp32, dequantised from the column-wise quantiser's own output."""
    import importlib
    import gcore_lowp as G
    L = importlib.import_module("gcore_lowp.grouped_gemm_fp8")
    m_splits, n_out = [513, 1400, 640, 0, 769, 1024, 600, 900, 700, 1025, 300, 513], 1408
    assert tile_rows(n_out, k_in, 11, 11) == tile
    g = torch.Generator(device="cuda").manual_seed(5)
    rows, E = sum(m_splits), len(m_splits)
    x = torch.randn(rows, k_in, generator=g, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn(E, n_out, k_in, generator=g, device="cuda", dtype=torch.bfloat16) * 0.02).requires_grad_(True)
    dy = torch.randn(rows, n_out, generator=g, device="cuda", dtype=torch.bfloat16) * 1e-3
    out = G.MyTeGroupedLinearFp8(E)(x, w, m_splits)
    dw, = torch.autograd.grad(out, w, dy)
    offs = L._offsets(m_splits, x.device)
    (xq, xs, nblk), (dq, ds, _) = L.quant_fp8_colwise_t(x, offs, m_splits, 128), L.quant_fp8_colwise_t(dy, offs, m_splits, 128)
    before = 0
    for e, nb in enumerate(nblk):
        if not nb:
            assert not dw[e].any()
            continue
        def operand(q, s, n):
            q = q.view(torch.float8_e4m3fn)[n * 128 * before:n * 128 * (before + nb)].view(n, 128 * nb)
            return deq(q, s.view(torch.float8_e8m0fnu)[n * before:n * (before + nb)].view(n, nb), 1)
        close(dw[e], operand(dq, ds, n_out) @ operand(xq, xs, k_in).t(), ("dW", e, m_splits[e]))
        before += nb
