"""The device-side tile schedule of the grouped GEMM with two tile heights (gemm_asm_grouped_mixed in
csrc/gemm_fp8_big.hip), restated on the host: from the rows per expert every workgroup derives its tiles (how both classes are
shared out: tests/test_grouped_balance_host.py) and for each its expert, its row tile and its column tile.  Over the grid the host
launches, every tile of every expert must come up exactly once, nothing else may come up, the grid bound must cover the
schedule, and the tiles an XCD runs together must belong to one expert or to neighbours.  A mistake here shows on the GPU as missing or doubly written output
rows, so it is checked where a mistake costs nothing.  Also the wide tile's weight-copy plan (256 x 288 loop)."""
import pytest

from tests.test_grouped_balance_host import share

CHUNK, GROUP_M = 32, 8


def classes(rows):
    rem = rows & 255
    return (rows >> 8) + (1 if rem > 128 else 0), (1 if 0 < rem <= 128 else 0)


def schedule(m_splits, N, grid):
    """-> list of (class, expert, local row tile, column tile, XCD, position in the XCD's run of the class) of every tile a workgroup takes."""
    tiles_n = -(-N // 256)
    cnts = {"big": [classes(r)[0] for r in m_splits], "small": [classes(r)[1] for r in m_splits]}
    out = []
    for xcd, big, small in share(sum(cnts["big"]) * tiles_n, sum(cnts["small"]) * tiles_n, grid):
        for cls, numbers in (("big", big), ("small", small)):
            for lin in numbers:
                gmt, incl = lin // tiles_n, 0
                for e, c in enumerate(cnts[cls]):                       # the expert whose running count covers gmt
                    if incl <= gmt < incl + c:
                        break
                    incl += c
                in_e = lin - incl * tiles_n
                grp, in_grp = divmod(in_e, GROUP_M * tiles_n)
                gm = min(c - grp * GROUP_M, GROUP_M)
                gn = CHUNK // gm
                nblk, in_blk = divmod(in_grp, gm * gn)
                out.append((cls, e, grp * GROUP_M + in_blk % gm, nblk * gn + in_blk // gm, xcd, lin))
    return out


CASES = {
    "zipf": None,                                           # the benchmark's rows per expert
    "ragged": [300, 0, 129, 128, 1, 255, 256, 257, 2048 + 130, 64, 0, 7146],
    "all_small": [5, 128, 77, 1],
    "all_big": [256, 512, 129, 3000],
    "one_heavy": [0, 0, 9000, 0],
    "empty": [0, 0, 0],
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("grid", [0, 8, 256, 304])
@pytest.mark.parametrize("N", [4096, 7168, 256, 4224, 128])
def test_every_tile_exactly_once(name, grid, N):
    """grid 0: a workgroup per tile, as the host launches where there are fewer tiles than CUs or the CUs are not known"""
    if CASES[name] is None:
        from tests._inputs import zipf_m_splits
        m_splits = zipf_m_splits().tolist()
    else:
        m_splits = CASES[name]
    tiles_n = -(-N // 256)
    bound = (sum(m_splits) // 256 + len(m_splits)) * tiles_n                         # mixed_grid: tiles of both classes at most
    assert sum(sum(classes(r)) for r in m_splits) * tiles_n <= bound
    got = schedule(m_splits, N, min(grid or 1 << 30, -(-bound // 8) * 8))
    want = set()
    for e, r in enumerate(m_splits):
        b, s = classes(r)
        for tn in range(tiles_n):
            want |= {("big", e, m, tn) for m in range(b)} | {("small", e, 0, tn) for _ in range(s)}
    tiles = [g[:4] for g in got]
    assert len(tiles) == len(set(tiles)), "a tile is handed out twice"
    assert set(tiles) == want
    # rows covered: big tiles take 256 rows each from the expert's start, the small tile what is left after them
    for e, r in enumerate(m_splits):
        b, s = classes(r)
        covered = min(r, b * 256) + (r - (r >> 8) * 256 if s else 0)
        assert covered == r, (e, r, b, s)


@pytest.mark.parametrize("mine", [0, 1, 255, 256, 257, 1000])
@pytest.mark.parametrize("lead", [0, 1, 300])
def test_table_walk_of_a_workgroup(mine, lead):
    """A workgroup's tiles are looked up 256 at a time, one per thread: first the `lead` tiles of one class, then the other's, every
    position exactly once."""
    K_TABLE, seen = 256, []
    lead = min(lead, mine)
    for first in range(0, mine, K_TABLE):
        for t in range(K_TABLE):
            at = first + t
            if at < mine:
                seen.append((at >= lead, at if at < lead else at - lead))
    assert seen == [(False, k) for k in range(lead)] + [(True, k) for k in range(mine - lead)]


def test_an_xcd_runs_neighbouring_tiles_together():
    """32 consecutive tiles of an XCD's run of a class, which its workgroups take at the same time: at most three experts, and for an
    expert with at least 8 row tiles a block of 8 x 4."""
    from tests._inputs import zipf_m_splits
    got = schedule(zipf_m_splits().tolist(), 4096, 256)
    by, start = {}, {}
    for cls, e, m, tn, xcd, lin in got:
        start[cls, xcd] = min(lin, start.get((cls, xcd), lin))
    for cls, e, m, tn, xcd, lin in got:
        by.setdefault((cls, xcd, (lin - start[cls, xcd]) // CHUNK), []).append((e, m, tn))
    for (cls, xcd, chunk), tiles in by.items():
        experts = {t[0] for t in tiles}
        assert len(experts) <= 3, (cls, xcd, chunk, experts)           # 16 column tiles per row tile: 32 numbers span <= 3 experts
        if len(experts) == 1 and cls == "big":
            ms, ns = {t[1] for t in tiles}, {t[2] for t in tiles}
            assert len(ms) * len(ns) >= len(tiles)                     # a rectangle of row x column tiles, not a line of 32


def test_wide_tile_weight_copy_plan():
    """256 x 288 loop: copy i of wave w moves the group of 8 weight rows WIDE_GROUP[i] + w (the fifth copy: waves 0..3,
    groups 16, 17, 34, 35).  The 36 groups must each be moved once; the mid-step part must be exactly the first 64
    rows of both wave columns; every group of a wave must have the wave's parity (one swizzled source offset serves all)."""
    group = (0, 18, 8, 26)
    moved, mid = [], []
    for w in range(8):
        mine = [g + w for g in group] + ([(16 if w < 2 else 32) + w] if w < 4 else [])
        assert all(g % 2 == w % 2 for g in mine)
        moved += mine
        mid += mine[:2]
    assert sorted(moved) == list(range(36))
    rows_mid = sorted(r for g in mid for r in range(8 * g, 8 * g + 8))
    assert rows_mid == list(range(0, 64)) + list(range(144, 208))


def test_weight_gradient_padding_and_launch_split():
    """Host side of the grouped weight gradient: blocks of 128 rows per expert under each padding rule (the rule the
    column-wise quantiser applies on the device), and the deal of the problems to kernels: every problem with K blocks in
    exactly one table, each table's K block counts multiples of what the launch promises, the running offsets those of
    the operands' layout, problems without rows listed apart."""
    pytest.importorskip("torch")
    from gcore_lowp import _abi as A
    from gcore_lowp.grouped_gemm_fp8 import choose_colwise_pad, padded_blocks, rowscale_launches
    rows = [0, 1, 128, 129, 256, 257, 512, 513, 1024, 1025, 7163]
    assert [padded_blocks(r, 128) for r in rows] == [0, 1, 1, 2, 2, 3, 4, 5, 8, 9, 56]
    assert [padded_blocks(r, 256) for r in rows] == [0, 2, 2, 2, 2, 4, 4, 6, 8, 10, 56]
    assert [padded_blocks(r, 512) for r in rows] == [0, 4, 4, 4, 4, 4, 4, 8, 8, 12, 56]
    assert [padded_blocks(r, A.PAD_MIXED) for r in rows] == [0, 1, 1, 2, 2, 4, 4, 8, 8, 12, 56]
    assert choose_colwise_pad(rows) == A.PAD_MIXED
    for k_blocks, whole in (([4, 1, 0, 8, 3, 12, 0, 5, 2, 1, 2], 1), ([4, 1, 0, 8, 16, 12, 0, 4, 2, 1, 2], 4), ([0, 0], None), ([2], None)):
        launches, empty = rowscale_launches(k_blocks)
        assert empty == [e for e, kb in enumerate(k_blocks) if kb == 0]
        seen = {}
        for table, multiple in launches:
            assert table and multiple in (1, 2, 4)
            for e, kb, before, zero in table:
                assert e not in seen and kb == k_blocks[e] and kb % multiple == 0 and zero == 0
                assert before == sum(k_blocks[:e])
                seen[e] = table
        assert sorted(seen) == [e for e, kb in enumerate(k_blocks) if kb]
        # one launch a kind at most: the problems of one K block, those of two, and the looped ones, longest first, with the promise
        # of whole groups of four exactly when all of them keep it
        kinds = [sorted({min(kb, 3) for _, kb, _, _ in table}) for table, _ in launches]
        assert all(len(k) == 1 for k in kinds) and len({k[0] for k in kinds}) == len(kinds)
        for table, multiple in launches:
            lengths = [kb for _, kb, _, _ in table]
            assert multiple == (min(lengths[0], 3) if lengths[0] < 3 else whole)
            assert lengths == sorted(lengths, reverse=True)
    # padding to 512 beyond 256 rows leaves whole groups of four only
    launches, _ = rowscale_launches([padded_blocks(r, A.PAD_MIXED) for r in range(0, 3000, 37)])
    assert all(m in (2, 4) or all(kb == 1 for _, kb, _, _ in t) for t, m in launches)
