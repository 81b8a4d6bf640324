"""The e8m0 loops that add every K block's product to the accumulators in fp32 (csrc/gen_gemm_loop.py: fold), walked on the host: the instructions one
wave executes, with the sums kept as lists of K blocks.  Every accumulator ends with every block once, no matrix instruction adds to
an earlier product, and a product is read only after the matrix instruction has had time to write it."""
import re

import pytest

from tests import test_gemm_loop_any_k_host as walk

gen = walk.gen
FOLD = {False: (128, 128, 2, 2, 1, True, 2, False, True, False, False, False, False, False, False, True),
        True: (128, 128, 2, 2, 1, True, 2, False, True, False, False, False, False, False, True, True)}


class Executed(list):
    """A program that notes the lines read from it."""

    def __init__(self, lines):
        super().__init__(lines)
        self.trace = []

    def __getitem__(self, i):
        self.trace.append(super().__getitem__(i))
        return self.trace[-1]


def executed(rag, kblocks):
    gen.configure(*FOLD[rag])
    gen.generate()
    lines = [ln.replace("%=", "") for ln in gen.lines]
    if rag:
        w = walk.Wave(lines, kblocks, 1, 0, 0)
        w.code = Executed(w.code)
        w.run()
        return w.code.trace
    start, end = lines.index("Lloop:"), lines.index("s_cbranch_scc1 Lloop")          # whole trips; no branch skips arithmetic
    return lines[:start] + lines[start:end + 1] * (kblocks // 4) + lines[end + 1:]


def span(t):
    lo, hi = re.match(r"v\[(\d+):(\d+)\]", t).groups()
    return range(int(lo), int(hi) + 1)


@pytest.mark.parametrize("rag,kblocks", [(True, n) for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 14, 23)] + [(False, n) for n in (4, 8, 20)])
def test_every_block_is_folded_once(rag, kblocks):
    acc, res, when, count, clock = {}, {}, {}, {}, 0
    for ln in executed(rag, kblocks):
        op, _, args = ln.partition(" ")
        a = [x.strip() for x in args.split(",")]
        clock += 1 + (int(a[0]) if op == "s_nop" else 0)
        if op.startswith("v_mfma"):
            assert a[3] == "0", ln
            block = count[a[0]] = count.get(a[0], -1) + 1
            for r in span(a[0]):
                assert r not in res, "a product is overwritten before it is added"
                res[r], when[r] = block, clock
        elif op == "v_add_f32":
            d, x, y = (int(t[1:]) for t in a)
            assert d == x and y == d - gen.ACC + gen.RES
            assert clock - when[y] > 12, ln                      # 8 passes of the matrix pipe: 11 wait states
            acc.setdefault(d, []).append(res.pop(y))
    assert not res and set(acc) == set(range(gen.ACC, gen.ACC + 64))
    assert all(v == list(range(kblocks)) for v in acc.values())
