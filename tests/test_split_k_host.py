"""Scratch of the dense GEMM's K ranges (lp_gemm_split_workspace_bytes): the partial sums of a plan's ranges and no more, and asked for only
where there is a K to cut."""
import random

import pytest


def test_split_scratch_is_bounded():
    from gcore_lowp import _abi
    L = _abi.lib()
    cap = L.lp_gemm_static_scratch_bytes()
    rng = random.Random(7)
    seen = 0
    for _ in range(4000):
        M, N, K = rng.randint(1, 8192), 128 * rng.randint(1, 144), 128 * rng.randint(1, 160)
        need = L.lp_gemm_split_workspace_bytes(M, N, K)
        tiles = (M + 127) // 128 * (N // 128)
        assert 0 <= need <= cap // 2, (M, N, K, need)
        if need:
            # a tile per workgroup of at most one round
            pieces, left = divmod(need, 128 * 128 * 4)
            assert left == 0 and 2 <= pieces <= 256 and tiles <= 800 and K >= 24 * 128, (M, N, K, need)
            seen += tiles > 32
    assert seen > 300
    assert L.lp_gemm_split_workspace_bytes(1, 4096, 7168) == 0 and L.lp_gemm_split_workspace_bytes(512, 4096, 1024) == 0
    assert [L.lp_gemm_split_workspace_bytes(*s) for s in ((0, 128, 128), (8, 100, 128), (8, 128, 100))] == [0, 0, 0]


@pytest.mark.parametrize("M,N,K", [(47, 6528, 6528), (33, 8192, 6144), (64, 6144, 7168), (64, 8192, 7168), (33, 8192, 8064), (43, 8192, 14464), (17, 6144, 7296), (22, 6016, 7424),
                                   (18, 5888, 13696), (24, 6144, 12032), (32, 5632, 9216), (23, 5376, 14336), (23, 5632, 18432), (65, 8192, 6144),
                                   (512, 2048, 5632), (64, 4096, 7168), (128, 4096, 5504)], ids=str)
def test_shapes_the_decode_kernels_are_faster_at_are_not_cut(M, N, K):
    from gcore_lowp import _abi
    assert _abi.lib().lp_gemm_split_workspace_bytes(M, N, K) == 0


@pytest.mark.parametrize("M,N,K", [(64, 5120, 6144), (56, 4224, 7168), (33, 5120, 7296), (44, 8192, 9216), (35, 7168, 16768), (24, 5120, 8192), (17, 5376, 14464), (24, 6144, 18432),
                                   (96, 8192, 6144), (65, 4096, 5632), (512, 2048, 6144)], ids=str)
def test_shapes_the_ranges_are_faster_at_are_cut(M, N, K):
    from gcore_lowp import _abi
    assert _abi.lib().lp_gemm_split_workspace_bytes(M, N, K) > 0


def test_scratch_by_type_of_scales():
    """Decode shapes ask for none with e8m0 scales, which keep the decode kernels; elsewhere both types take the same plan, of at most 256 pieces."""
    from gcore_lowp import _abi
    L = _abi.lib()
    for M, N, K in ((64, 5120, 6144), (48, 8192, 9216), (24, 5120, 9216), (70, 4096, 7168), (512, 1024, 7168), (64, 6144, 14336)):
        assert L.lp_gemm_split_workspace_bytes(M, N, K) > 0 == L.lp_gemm_block_workspace_bytes(_abi.E8M0, M, N, K), (M, N, K)
    for M, N, K in ((2048, 256, 8192), (4096, 128, 8192), (129, 128, 7168), (145, 2176, 12416), (1899, 3072, 13696)):
        need = L.lp_gemm_split_workspace_bytes(M, N, K)
        assert 0 < need <= 16 << 20 and need == L.lp_gemm_block_workspace_bytes(_abi.E8M0, M, N, K), (M, N, K)


def test_scratch_holds_whole_tiles_and_no_scale_copies():
    """42 tiles in six ranges; 512 rows at a K whose scales could be copied (to fp32, by a tuning aid that is off)."""
    from gcore_lowp import _abi
    L = _abi.lib()
    assert L.lp_gemm_split_workspace_bytes(24, 5376, 9216) == 6 * 128 * 5376 * 4
    assert L.lp_gemm_split_workspace_bytes(512, 512, 7168) == 8 * 512 * 512 * 4


def test_promised_workspace_takes_no_plan_it_does_not_promise():
    """Beyond 32 tiles lp_gemm_workspace_bytes has room for scale copies alone: less than the call wants for K ranges, however long K is."""
    from gcore_lowp import _abi
    L = _abi.lib()
    rng = random.Random(9)
    seen = 0
    for _ in range(20000):
        M, N, K = rng.randint(65, 8192), 128 * rng.randint(1, 800), 512 * rng.randint(6, 400)
        if (M + 127) // 128 * (N // 128) <= 32:
            continue
        need, promised = L.lp_gemm_split_workspace_bytes(M, N, K), L.lp_gemm_workspace_bytes(M, N, K)
        assert need == 0 or need > promised, (M, N, K, need, promised)
        seen += need == promised + 256
    assert seen


def test_promised_scratch_holds_every_plan():
    """Problems of at most 32 tiles: the partial sums of the best plan, M rows per range, fit what lp_gemm_workspace_bytes promises."""
    from gcore_lowp import _abi
    L = _abi.lib()
    rng = random.Random(8)
    r256 = lambda x: (x + 255) // 256 * 256
    seen = 0
    for _ in range(4000):
        M, N, K = rng.randint(65, 4096), 128 * rng.randint(1, 32), 128 * rng.randint(32, 160)
        best, promised = L.lp_gemm_split_workspace_bytes(M, N, K), L.lp_gemm_workspace_bytes(M, N, K)
        copies = r256(M * (K // 128) * 4) + r256((N // 128) * (K // 128) * 4) if K % 512 == 0 else 0
        if (M + 127) // 128 * (N // 128) > 32 or promised == copies:
            continue
        ranges, left = divmod(best, (M + 127) // 128 * 128 * N * 4)
        assert left == 0 and ranges * M * N * 4 <= promised - copies, (M, N, K)
        seen += 1
    assert seen > 200
