"""The loops of the GEMM kernels that take any number of K blocks (csrc/gen_gemm_loop.py: rag), walked on the host: the scalar
program of the generated text is executed for one wave -- bases, counters, branches, copy requests and counted waits -- and
checked for what the device cannot report: every request stays inside its operand and every scale inside its table, the
fragments of step k are read from a stage whose copies of block k have landed, there are exactly as many steps as blocks, and
every wave that stages scales other waves read writes every group of them to the right half of LDS, before the barrier behind
which it is read.  A wave none of whose activation rows exist stages nothing anybody reads, except with row-scaled weights,
whose scales the second half of the waves stages for the whole tile."""
import importlib.util
import os
import re

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
spec = importlib.util.spec_from_file_location("gen_gemm_loop", os.path.join(HERE, "..", "g-core-gh_amd", "csrc", "gen_gemm_loop.py"))
gen = importlib.util.module_from_spec(spec)
spec.loader.exec_module(gen)

LOOPS = {          # name -> configure arguments
    "big": (256, 256, 4, 2, 1, False, 2, False, True, False, True, True, False, False, True),
    "big e8m0": (256, 256, 4, 2, 1, True, 2, False, True, False, True, True, False, False, True),
    "mid": (128, 128, 2, 2, 1, False, 2, False, True, False, False, False, False, False, True),
    "mid e8m0": (128, 128, 2, 2, 1, True, 2, False, True, False, False, False, False, False, True),
    "flat": (128, 256, 2, 4, 1, False, 3, False, True, False, True, False, False, False, True),
    "flat e8m0": (128, 256, 2, 4, 1, True, 3, False, True, False, True, False, False, False, True),
    "big [K, N]": (256, 256, 4, 2, 1, True, 2, False, True, False, True, True, True, False, True),
    "mid row scales": (128, 128, 2, 2, 1, True, 2, True, True, False, False, False, False, False, True),
    "big row scales": (256, 256, 4, 2, 1, True, 2, True, True, False, True, True, False, False, True),
    "160 columns": (128, 160, 2, 2, 1, False, 2, False, True, True, False, False, False, False, True),
    "160 columns e8m0": (128, 160, 2, 2, 1, True, 2, False, True, True, False, False, False, False, True),
    "flat [K, N]": (128, 256, 2, 4, 1, True, 3, False, True, False, True, False, True, False, True),
}
ABASE, BBASE, SBASE, BSBASE = 0x1_0000_0000 - 256, 0x3_0000_0000 - 384, 0x5_0000_0001, 0x7_0000_0003     # low halves that carry
BSBASE2 = 0x9_0000_0005                                      # the second row of weight scales of a wave column that straddles two
NPITCH = 1408                                                # [K, N]: columns of the stored weight


class Wave:
    def __init__(self, lines, kblocks, copies, idle, second, wave=0, groups=20):
        g = gen
        self.wave, self.row_groups = wave, groups                # (160 columns: the groups of eight weight rows there are of the tile's 20)
        self.kblocks, self.copies, self.idle = kblocks, copies, idle
        self.code, self.labels = [], {}
        for ln in lines:
            if ln.endswith(":"):
                self.labels[ln[:-1]] = len(self.code)
            else:
                self.code.append(ln)
        ops = dict(klast=(kblocks - 1) * 128, krem=kblocks & 3, trips=(kblocks + 3) // 4, m0base=0, bsstride=NPITCH // 128,
                   bstep=128 * NPITCH, flags=copies | idle << 1 | second << 2 | (1 - second) << 3, bsbfe=0,
                   ard0=0, ard1=0, brd0=g.NSTAGE * g.A_BYTES, brd1=g.NSTAGE * g.A_BYTES)
        for i in range(8):
            ops[f"brdn{i}"] = ops["brd0"]
        if g.WIDE:
            ops.update(bstride=8 * 128 * kblocks, g4=8 if wave < 2 else 16, glim=groups - wave, splitnb=3)
        self.ops = ops
        self.pairs = dict(abase=ABASE, bbase=BBASE, sbase=SBASE, bsptr=BSBASE, bsptr2=BSBASE2)
        self.moved = {}                                          # 160 columns: group of LDS rows -> the groups of weight rows copied there
        self.s, self.v, self.scc, self.m0 = {}, {}, 0, 0
        self.queue, self.landed, self.scales_on_way = [], {}, None
        self.step, self.mfma, self.groups = 0, 0, []
        self.staged, self.unsettled, self.staging = [], False, []        # LDS halves written; a write not waited for; the instructions on staged scales

    def val(self, t):
        t = t.strip()
        if t.startswith("%["):
            return self.ops[t[2:-1]]
        if t == "m0":
            return self.m0
        if re.fullmatch(r"s\d+", t):
            return self.s[int(t[1:])]
        if re.fullmatch(r"v\d+", t):
            return self.v.get(int(t[1:]), 0)
        return int(t, 0)

    def pair(self, t):
        lo = int(re.match(r"s\[(\d+)", t.strip()).group(1))
        return self.s[lo] | self.s[lo + 1] << 32

    def put(self, t, x):
        if t == "m0":
            self.m0 = x & 0xFFFFFFFF
        else:
            self.s[int(t[1:])] = x & 0xFFFFFFFF

    def request(self, what):
        self.queue.append(what)

    def settle(self, n):
        while len(self.queue) > n:
            kind, *rest = self.queue.pop(0)
            if kind == "copy":
                m0, block = rest
                self.landed[m0] = block
        # a group of scales may be used once none of its requests is on its way

    def in_flight(self, kind):
        return any(q[0] == kind for q in self.queue)

    def scale_request(self, text):
        g = gen
        m = re.match(r"(global_load_(?:ubyte|dwordx4|dword)|s_load_dword(?:x2|x4)?) \S+,? ?(.*)", text)
        op, rest = m.group(1), m.group(2)
        size = {"global_load_ubyte": 1, "global_load_dword": 4, "global_load_dwordx4": 16, "s_load_dword": 4, "s_load_dwordx2": 8,
                "s_load_dwordx4": 16}[op]
        base = self.pair(re.search(r"s\[\d+:\d+\](?=,| offset|$)", rest).group(0))
        off = re.search(r"offset:(\d+)", rest)
        off = int(off.group(1)) if off else int(rest.split(",")[-1], 0) if op.startswith("s_load") else 0
        ss = 1 if g.HW else 4
        for name, start, pitch in (("a", SBASE, 1), ("b", BSBASE, NPITCH // 128 if g.NN else 1), ("b2", BSBASE2, 1)):
            rel = base + off - start
            if 0 <= rel < 1 << 20:
                if name == "b" and g.NN:
                    assert size == 1 and rel % pitch == 0 and rel // pitch < self.kblocks, (text, rel)
                    first = rel // pitch
                    n = 1
                else:
                    assert rel % ss == 0 and rel + size <= self.kblocks * ss, (text, rel, size, self.kblocks)
                    first, n = rel // ss, size // ss
                self.groups += [(name, first + i) for i in range(n)]
                if not op.startswith("s_load"):
                    self.request(("scale",))
                return
        raise AssertionError((text, hex(base)))

    def run(self):
        g, pc, budget = gen, 0, 400000
        while pc < len(self.code):
            budget -= 1
            assert budget > 0, "the loop does not end"
            ln = self.code[pc]
            pc += 1
            op, _, args = ln.partition(" ")
            a = [x.strip() for x in args.split(",")]
            if op == "s_mov_b64":
                if a[0].startswith("s[") and a[1].startswith("%["):
                    lo, x = int(a[0][2:].split(":")[0]), self.pairs[a[1][2:-1]]
                    self.s[lo], self.s[lo + 1] = x & 0xFFFFFFFF, x >> 32
                elif a[0].startswith("s[") and a[1].startswith("s["):
                    lo, src = int(a[0][2:].split(":")[0]), int(a[1][2:].split(":")[0])
                    self.s[lo], self.s[lo + 1] = self.s.get(src, 0), self.s.get(src + 1, 0)
            elif op == "s_mov_b32":
                self.put(a[0], self.val(a[1]))
            elif op in ("s_add_u32", "s_addc_u32", "s_sub_u32"):
                x = self.val(a[1]) + self.val(a[2]) + self.scc if op == "s_addc_u32" else self.val(a[1]) + (self.val(a[2]) if op == "s_add_u32" else -self.val(a[2]))
                self.put(a[0], x)
                self.scc = int(x >> 32 != 0)
            elif op in ("s_and_b32", "s_xor_b32", "s_lshr_b32", "s_lshl_b32", "s_mul_i32"):
                x, y = self.val(a[1]), self.val(a[2])
                self.put(a[0], x << y if op == "s_lshl_b32" else {"s_and_b32": x & y, "s_xor_b32": x ^ y, "s_lshr_b32": x >> y, "s_mul_i32": x * y}[op])
            elif op == "s_bfe_u32":
                x, y = self.val(a[1]), self.val(a[2])
                self.put(a[0], x >> (y & 31) & (1 << (y >> 16)) - 1)
            elif op.startswith("s_cmp_"):
                x, y = self.val(a[0]), self.val(a[1])
                self.scc = int({"eq": x == y, "lg": x != y, "lt": x < y, "gt": x > y}[op.split("_")[2]])
            elif op == "s_bitcmp1_b32":
                self.scc = self.val(a[0]) >> self.val(a[1]) & 1
            elif op == "s_cselect_b32":
                self.put(a[0], self.val(a[1]) if self.scc else self.val(a[2]))
            elif op in ("s_cbranch_scc0", "s_cbranch_scc1", "s_branch"):
                if op == "s_branch" or self.scc == int(op[-1]):
                    pc = self.labels[a[0]]
            elif op == "global_load_lds_dwordx4":
                src = a[0][2:6]
                if src == "aoff":
                    rel = self.pair(a[1]) - ABASE
                    assert rel % 128 == 0 and 0 <= rel // 128 < self.kblocks, (ln, rel)
                    block = rel // 128
                elif g.WIDE:
                    rel = self.pair(a[1].split()[0]) - BBASE
                    group, block = rel // self.ops["bstride"], rel % self.ops["bstride"] // 128
                    # this wave's rows of the group lie inside the weight matrix; and the copy's place in LDS is that group's, or that of one past its end
                    assert rel % 128 == 0 and 0 <= group and group + self.wave < self.row_groups, (ln, group, block)
                    place = (self.m0 - g.NSTAGE * g.A_BYTES) % g.B_BYTES // 1024
                    assert place == group if place + self.wave < self.row_groups else group == 0, (ln, place, group)
                    self.moved.setdefault(place + self.wave, set()).add(block)
                else:
                    rel, unit = self.pair(a[1].split()[0]) - BBASE, 128 * NPITCH if g.NN else 128
                    assert rel % unit == 0 and 0 <= rel // unit < self.kblocks, (ln, rel)
                    block = rel // unit
                self.request(("copy", self.m0, block))
            elif op.startswith("global_load") or op.startswith("s_load"):
                self.scale_request(ln)
                self.staging.append(ln)
            elif op in ("v_mov_b32", "v_lshl_or_b32") and gen.HW and re.match(r"v1(1[2-9]|2[01])\b", a[0]):
                self.staging.append(ln)                      # registers of the scales on their way (e8m0 loops)
            elif op == "s_waitcnt":
                m = re.search(r"vmcnt\((\d+)\)", ln)
                if m:
                    self.settle(int(m.group(1)))
                if "lgkmcnt(0)" in ln:
                    self.unsettled = False
            elif op == "v_mov_b32" and a[1].startswith("%["):
                self.v[int(a[0][1:])] = self.ops.get(a[1][2:-1], 0)
            elif op == "v_add_u32" and a[2].startswith("%[") and a[2][2:-1] in self.ops:
                self.v[int(a[0][1:])] = self.val(a[1]) + self.val(a[2])
            elif op.startswith("ds_write"):
                # the group just written belongs to the trip after this one (to the first in the prologue)
                assert not self.in_flight("scale"), "scales are written to LDS while they are on their way"
                self.staged.append(self.s[54])
                self.unsettled = True
                self.staging.append(ln)
            elif op == "s_barrier":
                assert not self.unsettled, "a barrier with scales still on their way to LDS"
            elif op.startswith("ds_read_b128") or op.startswith("ds_read_b64_tr"):
                addr = self.val(a[-1].split()[0]) + int(re.search(r"offset:(\d+)", ln).group(1))
                is_a = addr < g.NSTAGE * g.A_BYTES
                stage = addr // g.A_BYTES if is_a else (addr - g.NSTAGE * g.A_BYTES) // g.B_BYTES
                lo, size = (stage * g.A_BYTES, g.A_BYTES) if is_a else (g.NSTAGE * g.A_BYTES + stage * g.B_BYTES, g.B_BYTES)
                want = self.step if (stage == self.step % g.NSTAGE) else self.step + 1
                mine = {m: b for m, b in self.landed.items() if lo <= m < lo + size}
                if want < self.kblocks and is_a:
                    # (of the weight rows a wave's own copies may be the half that is read later: counted in the waits' own test)
                    assert mine and all(b == want for b in mine.values()), (ln, want, mine)
                    assert not any(q[0] == "copy" and lo <= q[1] < lo + size and q[2] == want for q in self.queue), (ln, want)
            elif op.startswith("v_mfma"):
                self.mfma += 1
                if self.mfma % (g.NB * g.MB) == 0:
                    self.step += 1
        assert not self.queue, "requests are still out at the end"


@pytest.mark.parametrize("name", list(LOOPS))
def test_requests_stay_inside_and_every_block_is_multiplied_once(name):
    gen.configure(*LOOPS[name])
    gen.generate()
    lines = [ln.replace("%=", "") for ln in gen.lines]
    staging = {}
    ss_total = lambda kb: {("b", k) for k in range(kb)}
    for kblocks in (1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 14, 23):
        for copies in (0, 1):
            for second in (0, 1):
                for idle in ((0, 1) if gen.WITH_IDLE else (0,)):
                    w = Wave(lines, kblocks, copies, idle, second)
                    w.run()
                    if copies and (not idle or gen.BROW):
                        assert w.staged == [gen.SCL_HALF * (i & 1) for i in range((kblocks + 3) // 4)], (kblocks, idle, w.staged)
                        assert {x for x in w.groups if x[0] == "a"} == {("a", k) for k in range(kblocks)}
                    if gen.BROW:
                        staging.setdefault((kblocks, copies), []).append(w.staging)
                    if not idle:
                        assert w.step == kblocks and w.mfma == kblocks * gen.NB * gen.MB, (kblocks, w.step)
                        got = set(w.groups)
                        assert {x for x in got if x[0] == "b"} == (set() if gen.BROW else ss_total(kblocks)), (kblocks, sorted(got))
                        assert {x for x in got if x[0] == "a"} == ({("a", k) for k in range(kblocks)} if copies else set())
    if gen.WIDE:
        # all waves together: every group of weight rows there is at every block, wherever the matrix ends in the tile; the second row of scales like the first
        for kblocks in (1, 2, 5, 8, 23):
            for groups in (4, 8, 12, 16, 20):
                moved = {}
                for wave in range(4):
                    w = Wave(lines, kblocks, int(wave < 2), 0, int(wave >= 2), wave, groups)
                    w.run()
                    assert w.step == kblocks
                    assert {x for x in w.groups if x[0] == "b2"} == {("b2", k) for k in range(kblocks)}
                    for place, blocks in w.moved.items():
                        assert place not in moved, (place, wave)
                        moved[place] = blocks
                assert all(moved[i] == set(range(kblocks)) for i in range(groups)) and sorted(moved) == list(range(20)), (kblocks, groups, moved)
    for key, ways in staging.items():
        assert all(x == ways[0] for x in ways), ("an idle wave handles the scales it stages otherwise than a live one", key)
