"""The generated main loops of the 4-wave GEMM kernels, run instruction by instruction on the CPU for one wave (the four do the
same): every fragment read finds the k-block its stage's products want, landed and behind a barrier; no request overwrites a slot
that some wave may still read; every block is multiplied once, in ascending order."""
import importlib.util
import os
import re

import pytest

PATH = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "graph-compiler_amd", "csrc", "kernels", "gen_gemm_w4_mainloop.py")
spec = importlib.util.spec_from_file_location("gen_gemm_w4_mainloop", PATH)
G = importlib.util.module_from_spec(spec)
spec.loader.exec_module(G)

A_DMA, B_DMA, A_READ, B_READ = 0, 1 << 20, 0, 1 << 20  # where the rings start, in each address space of the model


class Wave:
    def __init__(self, c, pairs, tail_group):
        self.c, self.s, self.v, self.scc, self.m0 = c, {}, {}, 0, 0
        self.s.update({40: 0, 42: 0, 44: 64, 46: pairs, 47: A_DMA, 48: 0, 50: tail_group, 51: B_DMA})
        self.v.update({16: A_READ, 17: A_READ, **{20 + k: B_READ for k in range(4)}})
        self.now, self.waited, self.free = 0, 0, 0  # instruction counter; last lgkmcnt(0); the last one in front of a barrier
        self.queue = []       # requests in flight, in order
        self.lds = {}         # (operand, KiB of the wave's shares) -> [pair or k-block, landed, visible]
        self.last_read = {}   # (operand, slot) -> when
        self.mfmas, self.reads = 0, {}
        if tail_group:        # the set-up has put the first two pairs into both rings: a number of requests, the oldest, and zeros
            for op, n in (("a", c.mi), ("b", c.nb if c.tb else 2 * c.nb)):  # for the rest; the loop's requests start at pair 2
                for q in range(2):
                    for i in range(n):
                        cell = [q if op == "a" or c.tb else 2 * q + i // c.nb, len(self.queue) >= tail_group, False]
                        self.lds[op, q * n + i] = cell
                        if not cell[1]:
                            self.queue.append(cell)

    def val(self, x):
        return self.m0 if x == "m0" else self.s[int(x[1:])] if x[0] == "s" else int(x)

    def target(self, op):
        """Slot and KiB of this wave's share that m0 names; KiB of a share, slots."""
        c = self.c
        at, size = (self.m0, c.a_pair) if op == "a" else (self.m0 - B_DMA, c.b_pair if c.tb else c.b_block)
        return at // size, at % size // 1024, c.mi if op == "a" else c.nb, c.da if op == "a" else c.db * (1 if c.tb else 2)

    def request(self, op):
        c = self.c
        slot, i, unit, depth = self.target(op)
        assert 0 <= slot < depth and i < unit
        # what it brings: the address counts whole pairs (blocks of B stored [K,N]); those of the tail group come first
        step = 128 if op == "a" or c.tb else 64
        ptr = self.s[40 if op == "a" else 42]
        assert ptr % step == 0
        what = ptr // step + (0 if not self.s[50] else 2 if step == 128 else 4)
        read = self.last_read.get((op, slot))
        assert read is None or read < self.free, "a slot is overwritten that may still be read"
        cell = [what, False, False]
        self.lds[op, slot * unit + i] = cell
        self.queue.append(cell)

    def fragment(self, op, addr, offset, half):
        c = self.c
        block = self.mfmas // (c.mi * c.nj) + (1 if self.started else 0)
        addr -= A_READ if op == "a" else B_READ
        if op == "a" or c.tb:
            pair = c.a_pair if op == "a" else c.b_pair
            slot, n, want = (addr + offset) // pair, c.mi if op == "a" else c.nb, block // 2
            assert half == block % 2
        else:
            slot, n, want = (addr + offset) // c.b_block, c.nb, block
        for i in range(n):
            cell = self.lds[op, slot * n + i]
            assert cell[0] == want and cell[2], (op, block, cell)
        self.last_read[op, slot] = self.now
        self.reads.setdefault(block, 0)
        self.reads[block] += 1

    def run(self, text):
        self.started = False
        text = [re.sub(r"%=", "", t) for t in text]
        labels = {t[:-1]: i for i, t in enumerate(text) if t.endswith(":")}
        pc = 0
        while pc < len(text):
            t = text[pc]
            pc += 1
            self.now += 1
            op, *args = re.split(r"[ ,]+", t)
            if t.endswith(":") or op in ("s_nop", "v_accvgpr_write_b32", "ds_write_b128", "v_xor_b32"):
                continue
            if op in ("s_add_u32", "s_sub_u32"):
                x = self.val(args[1]) + (1 if op == "s_add_u32" else -1) * self.val(args[2])
                if args[0] == "m0":
                    self.m0 = x
                else:
                    self.s[int(args[0][1:])] = x
            elif op == "s_addc_u32":
                pass
            elif op == "s_mov_b32":
                if args[0] == "m0":
                    self.m0 = self.val(args[1])
                else:
                    self.s[int(args[0][1:])] = self.val(args[1])
            elif op in ("s_cmp_eq_u32", "s_cmp_lg_u32"):
                self.scc = int((self.val(args[0]) == self.val(args[1])) == (op == "s_cmp_eq_u32"))
            elif op == "s_cselect_b32":
                self.s[int(args[0][1:])] = self.val(args[1] if self.scc else args[2])
            elif op == "s_cbranch_scc1":
                pc = labels[args[0]] if self.scc else pc
            elif op == "s_branch":
                pc = labels[args[0]]
            elif op == "v_mov_b32":
                self.v[int(args[0][1:])] = self.v[int(args[1][1:])]
            elif op == "v_add_u32":
                self.v[int(args[0][1:])] = self.val(args[1]) + self.v[int(args[2][1:])]
            elif op == "s_waitcnt":
                m = re.search(r"vmcnt\((\d+)\)", t)
                if m:
                    assert int(m.group(1)) <= 63
                    while len(self.queue) > int(m.group(1)):
                        self.queue.pop(0)[1] = True
                if "lgkmcnt(0)" in t:
                    self.waited = self.now
            elif op == "s_barrier":
                self.free = self.waited
                for cell in self.lds.values():
                    cell[2] = cell[1]
            elif op == "global_load_lds_dwordx4":
                which = "a" if "s[40:41]" in t else "b"
                assert int(args[0][1:]) == (0 if which == "a" else 8) + self.target(which)[1]
                self.request(which)
            elif op.startswith("ds_read"):
                reg, off = int(re.search(r"\], v(\d+)", t).group(1)), int(re.search(r"offset:(\d+)", t).group(1))
                if op == "ds_read_b128":
                    self.fragment("a" if reg < 20 else "b", self.v[reg], off, (reg - 18) % 2 if reg < 20 else reg - 24)
                else:
                    self.fragment("b", self.v[reg], off, None)
            elif op.startswith("v_mfma"):
                self.started = True
                self.mfmas += 1
            else:
                raise AssertionError("instruction unknown to the model: " + t)


@pytest.mark.parametrize("c", G.CONFIGS, ids=lambda c: c.name)
@pytest.mark.parametrize("pairs", [2, 4, 6, 8, 10, 22, 64])
@pytest.mark.parametrize("tail_group", [0, 1, 10 ** 6])  # an incomplete group in front: one request of it, all of them
def test_every_read_finds_its_block(c, pairs, tail_group):
    fill, main = G.gen(c)
    w = Wave(c, pairs, tail_group)
    w.run(fill)
    w.run(main)
    assert w.mfmas == 2 * pairs * c.mi * c.nj and not w.queue
    per = c.mi + (c.nj if c.tb else 2 * c.nj)
    assert w.reads == {b: per for b in range(2 * pairs)}
    assert w.lds and max(cell[0] for (op, _), cell in w.lds.items() if op == "a") == pairs - 1
