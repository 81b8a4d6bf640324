"""How grouped launches share their tiles, restated on the host.  Two tile heights (gemm_asm_grouped_mixed in
csrc/gemm_fp8_big.hip): every tile of both classes is taken by exactly one workgroup of the XCD whose run it lies in, and no
workgroup has more work than a longest-first list schedule would give it: at most one small tile above the least loaded one of
its XCD (a big tile counts 3, a small one 2).  Lists of problems of one shape (list_coords in csrc/gemm_common.h): every tile
once, dealt to the XCDs in turn.  Problems of two K blocks (gemm_rowscale_strip in csrc/gemm_rowscale_small.hip): every tile once,
and a workgroup for every CU where there are tiles for it."""
import pytest


def share(all_big, all_small, grid):
    """-> per workgroup (XCD, big tile numbers, small tile numbers)"""
    out = []
    for b in range(grid):
        P, x, wg = grid >> 3, b & 7, b >> 3
        eb, es = all_big & 7, all_small & 7
        first_big, n_big = x * (all_big >> 3) + min(x, eb), (all_big >> 3) + (x < eb)
        first_small, n_small = x * (all_small >> 3) + max(0, x - (8 - es)), (all_small >> 3) + (x >= 8 - es)
        rounds, r = divmod(n_big, P)
        extra = wg < r
        shift = 2 * (P - r) + wg if extra else wg - 2 * r
        zeroth = shift if extra else wg - r
        mine_small = 0
        if zeroth < n_small:
            rest = n_small - shift
            mine_small = 1 + ((rest - 1) // P if rest > P else 0)
        big = [first_big + k * P + wg for k in range(rounds + extra)]
        small = [first_small + (zeroth if k == 0 else k * P + shift) for k in range(mine_small)]
        out.append((x, big, small))
    return out


@pytest.mark.parametrize("grid", [8, 16, 256, 304])
@pytest.mark.parametrize("all_small", [0, 1, 7, 9, 31, 32, 255, 416, 513, 2048, 5000])
def test_every_tile_once_and_balanced(grid, all_small):
    for all_big in (0, 1, 8, 63, 64, 160, 255, 256, 257, 300, 1000, 3333):
        got = share(all_big, all_small, grid)
        assert sorted(t for _, b, _ in got for t in b) == list(range(all_big)), (all_big, all_small, grid)
        assert sorted(t for _, _, s in got for t in s) == list(range(all_small)), (all_big, all_small, grid)
        for x in range(8):
            load = [(3 * len(b) + 2 * len(s), len(s)) for xx, b, s in got if xx == x]
            least = min(w for w, _ in load)
            assert all(w - 2 <= least for w, small in load if small), (all_big, all_small, grid, load)
            runs = [t for xx, b, _ in got if xx == x for t in b]
            assert not runs or max(runs) - min(runs) + 1 == len(runs)          # one run of numbers per XCD


def list_tiles(G, tiles_m, tiles_n, slots):
    """list_shift, list_grid and list_coords of csrc/gemm_common.h -> tiles in a piece, per XCD the (problem, tile number) of its workgroups"""
    tiles, chunks = tiles_m * tiles_n, -(-G * tiles_m * tiles_n // 32)
    most = -(-chunks // 8)
    alike = most * 8 * 4 <= chunks * 5
    piece = 32 if alike or slots and chunks >= 8 and -(-most * 32 // slots) <= -(-G * tiles // (8 * slots)) else 8
    out = [[] for _ in range(8)]
    for b in range(-(-(G * tiles) // (8 * piece)) * 8 * piece):
        s, xcd = b >> 3, b & 7
        turn = s // piece
        g, lin = divmod((turn * 8 + (7 - xcd if turn % 2 else xcd)) * piece + s % piece, tiles)
        if g < G:
            out[xcd].append((g, lin))
    return piece, out


@pytest.mark.parametrize("G", [1, 2, 3, 15, 20, 32, 64])
@pytest.mark.parametrize("tiles_m,tiles_n", [(1, 1), (2, 2), (4, 4), (4, 6), (6, 8), (8, 8), (8, 11), (11, 16), (9, 23), (16, 16), (32, 32)])
@pytest.mark.parametrize("slots", [0, 64])
def test_problem_lists_cover_every_tile_once_on_all_xcds(G, tiles_m, tiles_n, slots):
    piece, per_xcd = list_tiles(G, tiles_m, tiles_n, slots)
    assert sorted(t for x in per_xcd for t in x) == [(g, lin) for g in range(G) for lin in range(tiles_m * tiles_n)]
    # a deal in turn: no XCD has more than its share of all tiles and one piece more
    assert max(map(len, per_xcd)) <= G * tiles_m * tiles_n / 8 + piece


def strips(G, tiles_m, tiles_n):
    """launch_rowscale_small and gemm_rowscale_strip -> strip length, per XCD the (problem, row tile, column tiles) of its workgroups"""
    cuts = [s for s in range(1, min(8, tiles_n) + 1) if -(-tiles_n // -(-tiles_n // s)) == s]
    strip = min(cuts, key=lambda s: (-(-G * tiles_m * -(-tiles_n // s) // 512) * (s + 2), -s))
    runs = tiles_m * -(-tiles_n // strip)
    piece = 8
    while piece > 1 and -(-G * runs // piece) < 8:
        piece //= 2
    out = [[] for _ in range(8)]
    for b in range(-(-G * runs // (8 * piece)) * 8 * piece):
        in_xcd, xcd = b >> 3, b & 7
        g, run = divmod((in_xcd // piece * 8 + xcd) * piece + in_xcd % piece, runs)
        if g < G:
            first = run // tiles_m * strip
            out[xcd].append((g, run % tiles_m, range(first, min(first + strip, tiles_n))))
    return strip, out


@pytest.mark.parametrize("G", [1, 2, 4, 8, 15, 40])
@pytest.mark.parametrize("tiles_m,tiles_n", [(1, 1), (1, 8), (3, 3), (4, 8), (8, 8), (11, 8), (11, 16), (16, 16), (9, 23), (32, 32), (56, 32)])
def test_strips_cover_every_tile_once_and_fill_the_chip(G, tiles_m, tiles_n):
    strip, per_xcd = strips(G, tiles_m, tiles_n)
    tiles = [(g, m, n) for x in per_xcd for g, m, ns in x for n in ns]
    assert sorted(tiles) == [(g, m, n) for g in range(G) for m in range(tiles_m) for n in range(tiles_n)]
    busy = [len(x) for x in per_xcd]
    assert strip <= 8 and sum(busy) >= min(256, G * tiles_m * tiles_n)           # one workgroup per CU where there are tiles for it
    assert sum(1 for n in busy if n) == min(8, sum(busy))                        # one strip per XCD before any has more
    assert max(busy) <= sum(busy) / 8 + 8
