#!/usr/bin/env python3
"""Writes the main loops of the 4-wave GEMM kernels (w4_body of gemm_tile256.hpp) as gfx950 assembly text.

A wave owns MI x NJ tiles of 16 x 16 (8 x 8: the 256 x 256 workgroup tile; 8 x 4 and 6 x 4: 256 and 192 rows by 128 columns).
The loop keeps the accumulators, two sets of fragments and the LDS addresses in fixed registers and places every
instruction by hand: with one wave per SIMD nothing hides a stall, and the compiler's allocator does not hold 64
accumulator tiles plus four fragment sets without copies and spills.  The kernel's set-up (addresses, column parameters)
and its epilogue stay C++; this text is two `asm volatile` statements between them (FILL: the first requests; MAIN).

Memory layout.  K advances in pairs of k-blocks: a k-block is 64 bytes of K per row (one MFMA k-step for all tiles of the
wave), a pair is 128 bytes, a whole cache line.  An operand whose rows run along K (A; B stored [N,K]) is requested in
pairs: eight lanes fetch a row's 128 bytes.  (Requested block by block, every line went from L2 to the compute unit twice,
64 bytes of it used each time: 12.5 million line reads for bf16 4096^3 where 8.4 million hold the operands' tiles, 16.7
million with B stored [N,K].)  Its LDS ring has DA (DB) slots of one pair; in a slot row r lies at 128 r, its 16-byte chunk c
at chunk position c ^ (r / 2 % 8).  B stored [K,N] is requested block by block, its ring has 2 DB slots of one block, read
through the transposing LDS load.

Register contract with the kernel (inputs in fixed registers, see the constraint lists in gemm_tile256.hpp):
  v[0:MI-1]   A: byte offset of this lane inside a pair, per DMA instruction of the wave (MI per pair)
  v[8:..]     B: the same (NJ per pair stored [N,K]; NJ/2 per block stored [K,N])
  v16, v17    LDS address of this lane's A fragment of row tile 0 in slot 0, first / second block of the pair
  v[20:23]    B stored [N,K]: v20, v21 likewise; stored [K,N]: of column tiles 0, 2, 4, 6 in slot 0, first block
  v18, v19, v[24:27]  the same for the slot being read
  v28         LDS address at which this lane writes accumulator tile (0, 0) for the epilogue
  s[40:41]    A tile: address of the next pair to request;  s[42:43]  B tile: of the next pair / block
  s[44:45]    bytes from one block of B stored [K,N] to the next
  s46         pairs of k-blocks in all (even, at least 2)
  s47, s51    LDS address of this wave's share of slot 0 of A / of B (DMA target)
  s48         int8: 0x80808080 when A is u8 (the bytes are flipped to s8 on the way into the MFMA), else 0
  s49         scratch (keeps m0);  s52..s57 slot bookkeeping, scratch
  s50         not 0: the first two pairs are an incomplete group of K that the set-up puts into slots 0 and 1 itself
              (in front of FILL, its requests are the oldest), and s[40:43] point at the pair behind them.  MAIN waits for
              them, with its accumulators cleared meanwhile
  a[0:..]     out: accumulator tile (jt, it) = a[(jt*MI+it)*4 : +4]
  v[32:..]    A fragments (MI row tiles x 4 registers) of first / second blocks, then B fragments likewise

One stage = one k-block.  Stage t computes block t from registers; between its MFMAs it reads the fragments of block t+1
into the other set and requests what the ring has room for:
  a pair's slot is free once its second block is in registers, that is from the start of an odd stage on: the pair DA
  further on goes into it, spread over that stage and the next; a block's slot of B stored [K,N] is free a stage after it was
  read, and every stage requests the block 2 DB further on.
  s_waitcnt vmcnt(n) lgkmcnt(0); s_barrier in front of every stage that needs something new to be visible or may overwrite
  (with whole pairs on both sides: every second stage).  n comes from replaying the order of the requests (Plan below).
Requests are spread evenly over a stage (issued back to back the four waves' requests queue up in the address unit and stall
the waves: 8 % slower), fragment reads go one every 2 MFMAs from the second MFMA on (one per MFMA: 3 % slower), or as
closely as the stage needs, so that they have all returned long before it ends.
After the last stage the accumulators of column tiles 0-3 go to LDS for the epilogue (dump()).

8-bit operands with u8 activations: the A fragments of block t+1 are flipped to s8 (v_xor with 0x80808080) during stage t.
The A tiles are read first, and LDS returns data in order, so each tile's four flips sit behind a partial wait
(s_waitcnt lgkmcnt(n), n = the reads issued after that tile's) that has long been satisfied.
"""
import sys

DUMP_PITCH = 272  # W4_DUMP_PITCH of gemm_tile256.hpp


class Cfg:
    def __init__(self, name, es, tb, mi, nj, da, db):
        self.name, self.es, self.tb, self.mi, self.nj, self.da, self.db = name, es, tb, mi, nj, da, db
        self.bm, self.bn = 32 * mi, 32 * nj
        self.a_pair, self.b_pair = self.bm * 128, self.bn * 128
        self.b_block = self.b_pair // 2
        self.a_region = da * self.a_pair
        self.lds = self.a_region + db * self.b_pair
        assert self.lds <= 160 * 1024 and mi % 2 == 0 and nj % 2 == 0
        self.nb = nj if tb else nj // 2  # B requests of a wave per pair / per block
        self.af = [32, 32 + 4 * mi]
        self.bf = [32 + 8 * mi, 32 + 8 * mi + 4 * nj]
        self.vend = 32 + 8 * (mi + nj)
        # requests of a stage: (operand, how many of the unit's requests), odd stage then even stage
        if tb:
            if db < 3:  # B's pair must be on its way before the even stage
                self.odd, self.even = [("b", nj)], [("a", mi)]
            else:
                first = max(0, (mi + nj) // 2 - nj)
                self.odd, self.even = [("b", nj)] + ([("a", first)] if first else []), [("a", mi - first)]
        else:
            self.odd, self.even = [("b", self.nb), ("a", mi // 2)], [("a", mi // 2), ("b", self.nb)]
        self.look = max(da, db if tb else db + 1)  # the steady loop requests up to this many pairs ahead
        assert self.look <= 4


class Plan:
    """Replays the requests of a whole product of P pairs and says what each stage waits for."""

    def __init__(self, c, P):
        self.c, self.P = c, P
        order = []  # units in the order of their (last) request
        for q in range(max(c.da, c.db)):
            if q < min(c.da, P):
                order += [("a", q)] * c.mi
            if q < min(c.db, P):
                order += [("b", q)] * c.nb if c.tb else [("b", 2 * q)] * c.nb + [("b", 2 * q + 1)] * c.nb
        self.wait = []  # vmcnt per stage; None: nothing new needed
        self.fills = []  # per stage: [(operand, unit, first request, requests)]
        covered = -1
        for t in range(2 * P):
            need = [("a", (t + 1) // 2), ("b", (t + 1) // 2 if c.tb else t + 1)]
            if t + 1 < 2 * P and (t % 2 == 1 or not c.tb or t == 0):
                last = max(len(order) - 1 - order[::-1].index(u) for u in need)
                self.wait.append(len(order) - 1 - last)
            else:
                self.wait.append(None)
            fills = []
            if P > 2:
                u = (t - 1) // 2 if t % 2 else t // 2 - 1
                done_a = sum(n for o, n in c.odd if o == "a") if t % 2 == 0 else 0
                for o, n in (c.odd if t % 2 else c.even):
                    if o == "a":
                        unit, first, valid = u + c.da, done_a, u + c.da < P and u >= 0
                    elif c.tb:
                        unit, first, valid = u + c.db, 0, u + c.db < P and u >= 0
                    else:
                        unit, first = t + 2 * c.db, 0
                        valid = unit < 2 * P
                    if valid:
                        fills.append((o, unit, first, n))
                        order += [(o, unit)] * n
            self.fills.append(fills)


def gen(c):
    mfma = "v_mfma_f32_16x16x32_bf16" if c.es == 2 else "v_mfma_i32_16x16x64_i8"
    trd = "ds_read_b64_tr_b16" if c.es == 2 else "ds_read_b64_tr_b8"
    M = c.mi * c.nj
    tag = c.name
    out = []
    emit = out.append

    def load(op, i):
        return "global_load_lds_dwordx4 v%d, s[%s]" % (i if op == "a" else 8 + i, "40:41" if op == "a" else "42:43")

    def advance(op):
        if op == "a":
            return ["s_add_u32 s40, s40, 128", "s_addc_u32 s41, s41, 0"]
        if c.tb:
            return ["s_add_u32 s42, s42, 128", "s_addc_u32 s43, s43, 0"]
        return ["s_add_u32 s42, s42, s44", "s_addc_u32 s43, s43, s45"]

    def rotate(end):
        """Slot bookkeeping at the end of an even stage: the slot just read is the next to fill, the next one is read.
        s52, s54: offset of the slot being read (A, B); s53: DMA target of the A pair to come, s55: of the B pair or second
        block, s56: of the first block (stored [K,N])."""
        ins = ["s_add_u32 s53, s47, s52",
               "s_add_u32 s55, s51, s54"] + ([] if c.tb else ["s_add_u32 s55, s55, %d" % c.b_block])
        for reg, size, depth in (("s52", c.a_pair, c.da), ("s54", c.b_pair, c.db)):
            ins += ["s_add_u32 %s, %s, %d" % (reg, reg, size), "s_cmp_eq_u32 %s, %d" % (reg, size * depth), "s_cselect_b32 %s, 0, %s" % (reg, reg)]
        if not c.tb:
            ins += ["s_add_u32 s56, s51, s54"]
        ins += ["v_add_u32 v18, s52, v16", "v_add_u32 v19, s52, v17"]
        for k in range(2 if c.tb else c.nj // 2):
            ins += ["v_add_u32 v%d, s54, v%d" % (24 + k, 20 + k)]
        return ins

    def read_a(it, h):
        r = c.af[h] + 4 * it
        return ["ds_read_b128 v[%d:%d], v%d offset:%d" % (r, r + 3, 18 + h, it * 2048)]

    def read_b(jt, h):
        r = c.bf[h] + 4 * jt
        if c.tb:
            return ["ds_read_b128 v[%d:%d], v%d offset:%d" % (r, r + 3, 24 + h, jt * 2048)]
        off = h * c.b_block + (jt & 1) * 16 * c.es
        return ["%s v[%d:%d], v%d offset:%d" % (trd, r, r + 1, 24 + jt // 2, off),
                "%s v[%d:%d], v%d offset:%d" % (trd, r + 2, r + 3, 24 + jt // 2, off + 8 * c.bn)]

    def all_reads(h):
        """the fragment reads of one block in the order its MFMAs want them"""
        rd = []
        if c.es == 2:
            rd += read_b(0, h)
        for it in range(c.mi):  # (8-bit: the A tiles first, they are the ones the byte flips wait for)
            rd += read_a(it, h)
        for jt in range(1 if c.es == 2 else 0, c.nj):
            rd += read_b(jt, h)
        return rd

    def xor_tile(it, h):
        return ["v_xor_b32 v%d, s48, v%d" % (c.af[h] + 4 * it + k, c.af[h] + 4 * it + k) for k in range(4)]

    def stage(t, wait, fills, nxt, turn, loop_tail=None):
        """t: the stage (its parity counts); wait: vmcnt or None; turn: slot bookkeeping at the end"""
        h = t & 1
        barrier = nxt and (h == 1 or not c.tb)
        if wait is not None:
            emit("s_waitcnt vmcnt(%d) lgkmcnt(0)" % wait)
        else:
            emit("s_waitcnt lgkmcnt(0)")
        if barrier:
            emit("s_barrier")
        extras = [[] for _ in range(M)]
        pre = []
        dma = []  # (m0, load)
        for o, unit, first, n in fills:
            base = "s53" if o == "a" else "s55" if c.tb or h else "s56"
            for i in range(first, first + n):
                dma.append((["s_add_u32 m0, %s, %d" % (base, i * 1024)], [load(o, i)]))
            if o == "b" or first + n == c.mi:
                dma[-1][1].extend(advance(o))
        if dma:
            at = [i * M // len(dma) for i in range(len(dma))]
            pre += dma[0][0]
            for i, (m0, ld) in enumerate(dma):
                extras[at[i]] += ld
                if i:
                    extras[at[i] - 1] += m0
        last_read = 0
        if nxt:
            rd = all_reads(h ^ 1)
            step = min(2.0, 0.75 * M / len(rd))
            at_rd = [1 + int(k * step) for k in range(len(rd))]
            for k, ins in enumerate(rd):
                extras[at_rd[k]].append(ins)
            last_read = at_rd[-1]
            if c.es == 1:
                per = 1 if M >= 8 * c.mi else 2  # flips per MFMA
                x0 = M - 4 * c.mi // per - (8 if per == 1 else 1)
                for it in range(c.mi):
                    p0 = x0 + it * 4 // per
                    issued = sum(1 for a in at_rd if a <= p0)
                    assert issued > it
                    dmas = len([1 for a in at if a <= p0]) if dma else 0  # should they count
                    extras[p0].append("s_waitcnt lgkmcnt(%d)" % max(0, min(15, issued - (it + 1) - dmas)))
                    for k, ins in enumerate(xor_tile(it, h ^ 1)):
                        extras[p0 + k // per].append(ins)
        if turn:
            ins = rotate(None)
            assert last_read + 1 < M - 2
            for k, x in enumerate(ins):  # behind the last read and the last request
                extras[min(M - 2, max(last_read, at[-1] if dma else 0) + 1 + k // 4)].append(x)
        if loop_tail:
            extras[M - 1] += ["s_sub_u32 s46, s46, 1", "s_cmp_lg_u32 s46, 0"]
        for ins in pre:
            emit(ins)
        for jt in range(c.nj):
            breg = c.bf[h] + 4 * jt
            for it in range(c.mi):
                acc = (jt * c.mi + it) * 4
                areg = c.af[h] + 4 * it
                emit("%s a[%d:%d], v[%d:%d], v[%d:%d], a[%d:%d]" % (mfma, acc, acc + 3, breg, breg + 3, areg, areg + 3, acc, acc + 3))
                for ins in extras[jt * c.mi + it]:
                    emit(ins)
        if loop_tail:
            emit("s_cbranch_scc1 %s" % loop_tail)

    # ---- FILL: the requests of the first pairs (s50: all but the first two)
    def request(op, slot_off, first=0):
        n = c.mi if op == "a" else c.nb
        for i in range(n):
            emit("s_add_u32 m0, %s, %d" % ("s47" if op == "a" else "s51", slot_off + i * 1024))
            emit("s_nop 0")
            emit(load(op, i))
        for ins in advance(op):
            emit(ins)

    emit("s_mov_b32 s49, m0")  # m0 carries the DMA's LDS address in here; the compiler's value is put back
    emit("s_cmp_lg_u32 s50, 0")
    emit("s_cbranch_scc1 .LW4_%s_TAILGROUP_%%=" % tag)
    for q in range(max(c.da, c.db)):
        if q == 2:
            emit(".LW4_%s_TAILGROUP_%%=:" % tag)
            emit("s_cmp_eq_u32 s46, 2")
            emit("s_cbranch_scc1 .LW4_%s_FILLED_%%=" % tag)
        if q < c.da:
            request("a", q * c.a_pair)
        if q < c.db:
            if c.tb:
                request("b", q * c.b_pair)
            else:
                request("b", q * c.b_pair)
                request("b", q * c.b_pair + c.b_block)
    emit(".LW4_%s_FILLED_%%=:" % tag)
    emit("s_mov_b32 m0, s49")
    fill, out = out, []
    emit = out.append

    # ---- MAIN
    L = c.look
    plans = {P: Plan(c, P) for P in range(2, 40, 2)}
    big = plans[38]
    # what a stage waits for: the least over all lengths (a short product has fewer requests behind what it waits for)
    steady = [min(p.wait[t] for P, p in plans.items() for t in range(1 + par, 2 * (P - L) + 1, 2) if P > L and p.wait[t] is not None)
              if any(w is not None for w in big.wait[5 + par:7 + par:2]) else None for par in (0, 1)]
    tails = []  # stages 2 (P - L) + 1 .. 2 P - 1
    for k in range(2 * L - 1):
        ws = [p.wait[2 * (P - L) + 1 + k] for P, p in plans.items() if P >= 4]
        assert all((w is None) == (ws[0] is None) for w in ws)
        tails.append(None if ws[0] is None else min(ws))

    emit("s_mov_b32 s49, m0")
    for r in range(4 * M):
        emit("v_accvgpr_write_b32 a%d, 0" % r)
    emit("s_mov_b32 s52, 0")
    emit("s_mov_b32 s54, 0")
    emit("v_mov_b32 v18, v16")
    emit("v_mov_b32 v19, v17")
    for k in range(2 if c.tb else c.nj // 2):
        emit("v_mov_b32 v%d, v%d" % (24 + k, 20 + k))
    if not c.tb:
        emit("s_mov_b32 s56, s51")
    emit("s_cmp_eq_u32 s46, 2")
    emit("s_cbranch_scc1 .LW4_%s_SHORT_%%=" % tag)

    def first_block(P):
        """wait for pair 0 (block 0), read its first fragments"""
        p = plans[P]
        order_len = sum(min(d, P) * n for d, n in ((c.da, c.mi), (c.db, c.nb if c.tb else 2 * c.nb)))
        done = c.mi + c.nb  # pair 0 of A, pair / block 0 of B come first
        emit("s_waitcnt vmcnt(%d) lgkmcnt(0)" % (order_len - done))
        emit("s_barrier")
        out.extend(all_reads(0))
        if c.es == 1:
            emit("s_waitcnt lgkmcnt(0)")
            for it in range(c.mi):
                out.extend(xor_tile(it, 0))

    def tail_group(behind):
        """an incomplete group's requests have landed; those FILL sent behind them may be in flight"""
        emit("s_cmp_eq_u32 s50, 0")
        emit("s_cbranch_scc1 .LW4_%s_WHOLE%d_%%=" % (tag, behind))
        emit("s_waitcnt vmcnt(%d)" % behind)
        emit(".LW4_%s_WHOLE%d_%%=:" % (tag, behind))

    behind = max(c.da - 2, 0) * c.mi + max(c.db - 2, 0) * c.nb * (1 if c.tb else 2)
    assert behind > 0
    tail_group(behind)
    first_block(38)
    w0 = min(p.wait[0] for P, p in plans.items() if P >= 4)
    stage(0, w0 if not c.tb else None, big.fills[0], True, True)
    emit("s_sub_u32 s46, s46, %d" % L)
    emit("s_cmp_eq_u32 s46, 0")
    emit("s_cbranch_scc1 .LW4_%s_TAIL_%%=" % tag)
    emit(".LW4_%s_LOOP_%%=:" % tag)
    for par in (0, 1):
        stage(5 + par, steady[par], big.fills[5 + par], True, par == 1, loop_tail=".LW4_%s_LOOP_%%=" % tag if par == 1 else None)
    emit(".LW4_%s_TAIL_%%=:" % tag)
    for k in range(2 * L - 1):
        t = 2 * (38 - L) + 1 + k
        last = t == 2 * 38 - 1
        stage(t, tails[k], big.fills[t], not last, t % 2 == 0 and not last)
    # the results of the last MFMAs must have been written before anything reads the accumulators, and every wave
    # must have taken its last fragments before the ring is overwritten with them
    emit(".LW4_%s_DONE_%%=:" % tag)
    emit("s_nop 15")
    emit("s_nop 15")
    emit("s_waitcnt vmcnt(0) lgkmcnt(0)")
    emit("s_barrier")
    out.extend(dump(c, 0))
    emit("s_branch .LW4_%s_END_%%=" % tag)
    emit(".LW4_%s_SHORT_%%=:" % tag)
    tail_group(0)
    first_block(2)
    for t in range(4):
        stage(t, plans[2].wait[t] if (t or not c.tb) else None, [], t < 3, t in (0, 2))
    emit("s_branch .LW4_%s_DONE_%%=" % tag)
    emit(".LW4_%s_END_%%=:" % tag)
    emit("s_mov_b32 m0, s49")
    return fill, out


def dump(c, half):
    """Accumulators of column tiles 4*half .. 4*half+3 to the wave's LDS region as a row-major block of 64 columns: tile
    (jt, it) holds rows 16*it.. and columns 16*(jt%4)..; v28 = the lane's address for tile (0, 0)."""
    out = []
    for jt in range(4 * half, min(c.nj, 4 * half + 4)):
        for it in range(c.mi):
            acc = (jt * c.mi + it) * 4
            out.append("ds_write_b128 v28, a[%d:%d] offset:%d" % (acc, acc + 3, it * 16 * DUMP_PITCH + (jt % 4) * 64))
    out.append("s_waitcnt lgkmcnt(0)")
    return out


CONFIGS = [
    Cfg("BF16_8x8", 2, False, 8, 8, 3, 2), Cfg("BF16_TB_8x8", 2, True, 8, 8, 3, 2), Cfg("I8_8x8", 1, False, 8, 8, 3, 2),
    Cfg("BF16_8x4", 2, False, 8, 4, 3, 3), Cfg("BF16_TB_8x4", 2, True, 8, 4, 3, 3), Cfg("I8_8x4", 1, False, 8, 4, 3, 3),
    Cfg("BF16_6x4", 2, False, 6, 4, 4, 3), Cfg("BF16_TB_6x4", 2, True, 6, 4, 4, 4), Cfg("I8_6x4", 1, False, 6, 4, 4, 3),
    Cfg("BF16_4x4", 2, False, 4, 4, 4, 3), Cfg("BF16_TB_4x4", 2, True, 4, 4, 4, 4), Cfg("I8_4x4", 1, False, 4, 4, 4, 3),
    Cfg("BF16_8x6", 2, False, 8, 6, 3, 2), Cfg("BF16_TB_8x6", 2, True, 8, 6, 3, 2),
]


def main():
    path = sys.argv[1]
    with open(path, "w") as f:
        f.write("// generated by gen_gemm_w4_mainloop.py -- do not edit\n")

        def macro(name, lines):
            f.write("#define %s \\\n" % name)
            f.write(" \\\n".join('  "%s\\n"' % ln for ln in lines))
            f.write("\n\n")

        for c in CONFIGS:
            fill, main_loop = gen(c)
            macro("GCMI_W4_FILL_%s" % c.name, fill)
            macro("GCMI_W4_ASM_%s" % c.name, main_loop)
        # depths of the rings: DA, DB of w4_body
        f.write("template <int ES, bool TB, int MI, int NJ> struct W4Ring;\n")
        for c in CONFIGS:
            f.write("template <> struct W4Ring<%d, %s, %d, %d> { static constexpr int DA = %d, DB = %d; };\n"
                    % (c.es, "true" if c.tb else "false", c.mi, c.nj, c.da, c.db))
        for mi, nj in sorted({(c.mi, c.nj) for c in CONFIGS}):
            c = next(c for c in CONFIGS if (c.mi, c.nj) == (mi, nj))
            if nj > 4:
                macro("GCMI_W4_ASM_DUMP_HI_%dx%d" % (mi, nj), dump(c, 1))
            regs = ["v18", "v19", "v24", "v25", "v26", "v27"] + ["v%d" % r for r in range(32, c.vend)] + ["a%d" % r for r in range(4 * mi * nj)]
            f.write("#define GCMI_W4_CLOBBERS_%dx%d %s\n" % (mi, nj, ", ".join('"%s"' % r for r in regs)))


if __name__ == "__main__":
    main()
