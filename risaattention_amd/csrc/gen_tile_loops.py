#!/usr/bin/env python3
"""Writes the hand-scheduled tile loops of the kernels gen_dense_loop.py does not cover: scaled
scores (the causal rule, scales of any sign), additive and boolean masks, 64-key tiles, head dim 64.
One `asm volatile` statement per program, operands included, as tile_loop_<name>.inc beside this file.

    python3 gen_tile_loops.py

A program walks the first `count` listed tiles of a query block and leaves the copies of the one
after them in flight; the C++ loop of attention_kernel.hpp, whose arithmetic it repeats in the same
order bit for bit, walks the rest.  The order of a tile is gen_dense_loop.py's (copies between the
score products, maxima, exponent arguments, exponentials around the value products, output update;
wave priorities 0, 1, 2, 0).  What bounds these loops is vector issue, so what they save over the
compiled ones is instructions: the compiler forms every copy's source offset again in every tile
(addresses kept over its loop would be spilled), here they stay in registers.

Score modes:
  raw      FMA of the raw score with its scale, maxima of the seeded integers (no mask, scale > 0)
  scaled   scaled score rounded first, as every masked or causal launch has it
Masks of the scaled mode:
  bias     additive row of a key-only mask, staged with the tile; a tile whose row is zero skips it
  f32      additive float mask, staged in LDS.  There is one mask tile for both stages: its rows are
           read into registers at the top of a tile, so that the next tile's copies have the whole
           tile to land (read where they are applied, the copies have only the output update and the
           next score product)
  lanes    boolean mask as wave-uniform 64-bit words, 16 of them at a time in scalar registers
"""
import argparse
import pathlib
import sys

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent))
from gen_dense_loop import Emitter, add64  # noqa: E402

FIRST_SGPR = 36     # the compiler keeps the registers below for the operands
SEED_BIAS = 2048    # the seed address register is 2 KiB ahead so that stage 1 stays within a 16-bit offset
LOG2E = "0x3fb8aa3b"
ROW_FLOOR = "0xc7435000"      # -50000
MINUS_U8_OFFSET = "0xc0ffd1be"  # -7.9943534
NEG_INF = "0xff800000"
POS_INF = "0x7f800000"


class Program:
    """Shape, registers and operands of one program."""

    def __init__(self, name, dim, keys, scaled, mask=None, listed=False, tight=False):
        """tight: within 128 registers, for four workgroups per compute unit.  Probabilities are formed
        and packed over the scores, the score seeds stand in accumulator and V fragment registers (16
        moves per tile; read from LDS instead, lists of two to four tiles are 2-4 % slower and long ones
        1 % faster), and values whose uses do not overlap share registers."""
        self.name, self.dim, self.keys, self.scaled, self.mask, self.listed = name, dim, keys, scaled, mask, listed
        self.tight = tight
        assert scaled or mask is None
        assert not tight or (dim == 64 and mask == "lanes")
        self.kk, self.cb, self.rb = dim // 32, dim // 32, keys // 32
        self.tile_bytes = dim * keys
        self.seed_region = 2 * self.tile_bytes
        self.bias_region = self.seed_region + dim * 4
        self.stage = self.bias_region + keys * 4
        self.mask_region = 2 * self.stage          # f32: one mask tile behind both stages
        self.copies = self.tile_bytes // 4096      # 1 KiB copies per wavefront, for K and for V
        self.k_offsets = 2 if dim == 128 else 1    # distinct lane shares of the K copies (swizzle period)
        self.v_offsets = 2 if keys == 128 else 1
        self.v_rows = 1024 // keys                 # V rows of one copy
        self.next_vgpr = 0
        take = self.take
        self.S = [take(16) for _ in range(self.rb)]
        self.M = take(32) if mask == "f32" else None
        self.ACC = [take(16) for _ in range(self.cb)]
        if tight:  # (right behind the accumulators, see SEEDS)
            self.VF = [take(4) for _ in range(self.cb)]
        self.O = [take(16) for _ in range(self.cb)]
        self.Q = [take(4) for _ in range(self.kk)]
        if not tight:
            self.VF = [take(4) for _ in range(self.cb)]
        self.PK = list(self.S) if tight else [take(4), take(4)]
        # seed block of the score products: registers of its own where they are free (no moves), else
        # the V fragment registers, free in that phase
        # (tight: K fragments fill the lower half of an accumulator; the upper half of the last one
        # and the V fragments are sixteen free registers in a row)
        roomy = keys == 64 and mask != "f32" and not tight
        self.SEEDS = take(16) if roomy else self.ACC[-1] + 8 if tight else self.VF[0]
        self.seeds_kept = roomy
        self.T = None if tight else [take(1) for _ in range(4)]
        self.sc0, self.sc1 = take(1), take(1)
        self.mx0 = self.sc0 if tight else take(1)  # (the maxima follow the last use of the scales)
        self.negm = None if scaled else take(1)
        # free in the phases that use them
        if tight:
            self.mx1 = self.tmp = self.sc1
        else:
            self.mx1, self.tmp = self.PK[1], self.PK[1] + 1
        self.tscale, self.mrun, self.dpart = take(1), take(1), take(1)
        self.rowsum, self.qscale, self.seedval = take(1), take(1), take(1)
        self.upper0, self.upper1 = (self.rowsum, self.tscale) if tight else (self.tmp, self.PK[1] + 2)
        self.lane16 = self.rowsum if tight else self.T[0]  # lane * 16, row copies
        self.ka = take(1) if mask == "f32" else None     # K fragment address of k-step 0; the others by xor
        self.KA = None if mask == "f32" else [take(1) for _ in range(self.kk)]
        if keys == dim and self.KA:
            self.VA = self.KA                            # rows of the same length: the same addresses
            self.va_shared = True
        else:
            self.VA = [take(1) for _ in range(self.rb)]
            self.va_shared = False
        self.seedaddr = take(1)
        self.KC = [take(1) for _ in range(self.k_offsets)]
        self.VC = [take(1) for _ in range(self.v_offsets)]
        if mask == "f32":
            self.maddr, self.mch, self.mrow = take(1), take(1), take(1)
        assert self.next_vgpr <= 255, (name, self.next_vgpr)  # v255 is left to the compiler
        # head dim 64: three wavefronts per SIMD, four of a tight program (and three registers for the compiler)
        assert dim == 128 or self.next_vgpr <= (125 if tight else 167), (name, self.next_vgpr)
        self.next_sgpr = FIRST_SGPR
        stake = self.stake
        if mask == "lanes":
            self.words = stake(32, 4)
        self.ks = stake(4, 4)
        self.kptr, self.vptr, self.sumptr, self.ksptr = stake(2), stake(2), stake(2), stake(2)
        self.count, self.lds, self.qs2, self.klds = stake(1), stake(1), stake(1), stake(1)
        self.halfmask, self.tmp_s, self.tmp2_s = stake(2), stake(2), stake(2)
        if listed:
            self.list, self.tnext, self.tafter, self.index, self.last = stake(2), stake(1), stake(1), stake(1), stake(1)
        if mask is not None:
            self.maskptr = stake(2)
        if mask == "lanes":
            self.words_at = stake(2)
        self.vstep = stake(1)
        if mask == "f32":
            self.mstep, self.mlds, self.klass = stake(1), stake(1), stake(1)
            self.pairs = [stake(2) for _ in range(4)]
        assert self.next_sgpr <= 102, (name, self.next_sgpr)

    def take(self, count):
        first = self.next_vgpr
        self.next_vgpr += count
        return first

    def stake(self, count, align=None):
        align = align or count
        self.next_sgpr = -(-self.next_sgpr // align) * align
        first = self.next_sgpr
        self.next_sgpr += count
        return first

    def v_region(self, stage):
        return stage * self.stage + self.tile_bytes


def pair(first):
    return f"s[{first}:{first + 1}]"


def load_words(e, p, tile):
    """lanes: the words of the first key block of a tile (256 bytes of words per tile)."""
    e.ins(f"s_lshl_b32 s{p.words_at}, s{tile}, 8")
    e.ins(f"s_add_u32 s{p.words_at}, s{p.maskptr}, s{p.words_at}")
    e.ins(f"s_addc_u32 s{p.words_at + 1}, s{p.maskptr + 1}, 0")
    e.ins(f"s_load_dwordx16 s[{p.words}:{p.words + 15}], {pair(p.words_at)}, 0x0")
    e.ins(f"s_load_dwordx16 s[{p.words + 16}:{p.words + 31}], {pair(p.words_at)}, 0x40")


def tile_body(e, p, stage, prio, label):
    """One tile held in LDS stage `stage`; its copies fill the other stage with the next tile."""
    other = stage ^ 1
    base = stage * p.stage
    e.comment(f"===== tile in stage {stage} =====")
    e.ins("s_waitcnt vmcnt(0) lgkmcnt(0)")  # own copies of this tile; scalar loads asked for a tile ago
    e.ins("s_barrier")
    e.ins(f"s_setprio {prio[0]}")
    if p.mask == "bias":
        # the row of additive terms, 16 bytes per lane: is any of them not zero?
        e.valu(f"v_mbcnt_lo_u32_b32 v{p.T[0]}, -1, 0", [p.T[0]])
        e.valu(f"v_and_b32_e32 v{p.T[0]}, {p.keys // 4 - 1}, v{p.T[0]}", [p.T[0]])
        e.ins(f"s_add_u32 s{p.tmp_s}, s{p.lds}, {SEED_BIAS}")
        e.valu(f"v_lshl_add_u32 v{p.T[0]}, v{p.T[0]}, 4, s{p.tmp_s}", [p.T[0]])
        e.ds_read(p.PK[0], p.T[0], base + p.bias_region - SEED_BIAS)
    if p.mask == "f32":
        for kk in range(p.kk):
            source = p.ka
            if kk:
                source = p.T[kk]
                e.valu(f"v_xor_b32_e32 v{source}, {kk * 32}, v{p.ka}", [source])
            for rb in range(p.rb):
                e.ds_read(p.ACC[kk] + rb * 4, source, base + rb * 32 * p.dim)
        for group in range(8):
            source = p.T[group & 3]
            e.valu(f"v_xor_b32_e32 v{source}, {group // 4 * 128 + group % 4 * 32}, v{p.maddr}", [source])
            e.ds_read(p.M + group * 4, source, 0)
    else:
        for kk in range(p.kk):
            for rb in range(p.rb):
                e.ds_read(p.ACC[kk] + rb * 4, p.KA[kk], base + rb * 32 * p.dim)
    shift = {64: 6, 128: 7}
    if p.listed:
        # sources of the next listed tile: bases of the head (with this wave's share) + tile * stride
        e.ins(f"s_mov_b32 s{p.tnext}, s{p.tafter}")
    if not p.seeds_kept:
        for r in range(16):
            e.valu(f"v_mov_b32_e32 v{p.SEEDS + r}, v{p.seedval}", [p.SEEDS + r])

    def source(pointer, bits, target):
        """Scalar pair `target`: where the next tile's data start."""
        if p.listed:
            e.ins(f"s_lshl_b32 s{target}, s{p.tnext}, {bits}")
            e.ins(f"s_add_u32 s{target}, s{pointer}, s{target}")
            e.ins(f"s_addc_u32 s{target + 1}, s{pointer + 1}, 0")
        else:
            e.ins(f"s_mov_b64 {pair(target)}, {pair(pointer)}")

    def k_copy(i):
        def emit():
            if i == 0:
                source(p.kptr, shift[p.keys] + shift[p.dim], p.tmp2_s)
            e.ins(f"s_add_u32 m0, s{p.klds}, {other * p.stage + i * 1024}")
            e.ins("s_nop 0")
            # (no instruction offset: the hardware would add it to the LDS address as well)
            e.ins(f"global_load_lds_dwordx4 v{p.KC[i % p.k_offsets]}, {pair(p.tmp2_s)}")
            if i < p.copies - 1:
                add64(e, p.tmp2_s, 1024)
        return emit

    def v_copy(i):
        def emit():
            if i == 0:
                source(p.vptr, shift[p.keys], p.tmp_s)
            e.ins(f"s_add_u32 m0, s{p.klds}, {p.v_region(other) + i * 1024}")
            e.ins("s_nop 0")
            e.ins(f"global_load_lds_dwordx4 v{p.VC[i % p.v_offsets]}, {pair(p.tmp_s)}")
            if i < p.copies - 1:
                e.ins(f"s_add_u32 s{p.tmp_s}, s{p.tmp_s}, s{p.vstep}")
                e.ins(f"s_addc_u32 s{p.tmp_s + 1}, s{p.tmp_s + 1}, 0")
        return emit

    def row_copy(wave, lanes, region, pointer, bits, name):
        """16 bytes per lane by the first lanes of one wavefront."""
        def emit():
            e.ins(f"s_sub_u32 s{p.tmp_s}, s{p.klds}, s{p.lds}")
            e.ins(f"s_cmp_lg_u32 s{p.tmp_s}, {wave * p.copies * 1024}")
            e.ins(f"s_cbranch_scc1 {label}_{name}")
            source(pointer, bits, p.tmp_s)
            e.ins(f"s_mov_b64 exec, {hex((1 << lanes) - 1)}")
            e.ins(f"s_add_u32 m0, s{p.lds}, {other * p.stage + region}")
            e.ins("s_nop 0")
            e.ins(f"v_mbcnt_lo_u32_b32 v{p.lane16}, -1, 0")
            e.ins(f"v_lshlrev_b32_e32 v{p.lane16}, 4, v{p.lane16}")
            e.ins(f"global_load_lds_dwordx4 v{p.lane16}, {pair(p.tmp_s)}")
            e.ins("s_mov_b64 exec, -1")  # (every wavefront of the kernel runs with all its lanes)
            e.raw(f"{label}_{name}:")
        return emit

    def mask_copies():
        """f32: this wavefront's 32 rows of the next tile, over the rows it has just read."""
        for group in range(8):
            e.wait_lds(p.M + group * 4)
        e.ins(f"s_cmp_eq_u32 s{p.count}, 1")   # the tile behind the walk reads its mask elsewhere
        e.ins(f"s_cbranch_scc1 {label}_nomask")
        e.ins(f"s_mov_b64 {pair(p.tmp_s)}, {pair(p.maskptr)}")
        for i in range(8):
            register = p.T[i & 3]
            e.ins(f"s_movk_i32 s{p.tmp2_s}, {(i & 3) * 64}")
            e.valu(f"v_xad_u32 v{register}, v{p.mch}, s{p.tmp2_s}, v{p.mrow}", [register])
            e.ins(f"s_add_u32 m0, s{p.mlds}, {i * 1024}")
            e.ins("s_nop 0")
            e.ins(f"global_load_lds_dwordx4 v{register}, {pair(p.tmp_s)}")
            if i < 7:
                e.ins(f"s_add_u32 s{p.tmp_s}, s{p.tmp_s}, s{p.mstep}")
                e.ins(f"s_addc_u32 s{p.tmp_s + 1}, s{p.tmp_s + 1}, 0")
        e.raw(f"{label}_nomask:")

    copies = [k_copy(i) for i in range(p.copies)] + [v_copy(i) for i in range(p.copies)]
    copies.append(row_copy(0, p.dim // 4, p.seed_region, p.sumptr, shift[p.dim] + 2, "noseed"))
    if p.mask == "bias":
        copies.append(row_copy(1, p.keys // 4, p.bias_region, p.maskptr, shift[p.keys] + 2, "nobias"))
    products = p.kk * p.rb
    per_product = -(-len(copies) // products)

    # ---- S^T = K Q^T -----------------------------------------------------------------------------
    for kk in range(p.kk):
        for rb in range(p.rb):
            e.wait_lds(p.ACC[kk] + rb * 4)
            if kk == 0:
                e.need_valu_result_for_mfma(range(p.SEEDS, p.SEEDS + 16))
            e.mfma(p.S[rb], p.ACC[kk] + rb * 4, p.Q[kk], p.SEEDS if kk == 0 else p.S[rb])
            for _ in range(per_product):
                if copies:
                    copies.pop(0)()
        # accumulator seeds of channel block kk into the registers this k-step has just left
        for b4 in range(4):
            e.ds_read(p.ACC[kk] + b4 * 4, p.seedaddr, base + p.seed_region - SEED_BIAS + kk * 128 + b4 * 32)
    while copies:
        copies.pop(0)()
    if p.mask == "f32":
        mask_copies()
    if not p.listed:
        add64(e, p.kptr, p.tile_bytes)
        add64(e, p.vptr, p.keys)
        add64(e, p.sumptr, p.dim * 4)
        if p.mask in ("f32", "bias"):
            add64(e, p.maskptr, p.keys * 4)

    # ---- K scales of this tile (scalar registers) -> score scales of this lane's two key groups ----
    e.ins(f"s_setprio {prio[1]}")
    for register, slot in ((p.upper0, 2), (p.upper1, 3), (p.sc0, 0), (p.sc1, 1)):
        e.valu(f"v_mov_b32_e32 v{register}, s{p.ks + slot}", [register])
    for register, upper in ((p.sc0, p.upper0), (p.sc1, p.upper1)):
        e.valu(f"v_cndmask_b32_e64 v{register}, v{register}, v{upper}, {pair(p.halfmask)}", [register])
    for register in (p.sc0, p.sc1):
        e.valu(f"v_mul_f32_e32 v{register}, v{p.qscale}, v{register}", [register])
    for register in (p.sc0, p.sc1):
        e.valu(f"v_mul_f32_e32 v{register}, s{p.qs2}, v{register}", [register])

    scores = [p.S[rb] + i for rb in range(p.rb) for i in range(16)]
    scale_of = lambda i: p.sc1 if i & 2 else p.sc0
    if p.mask == "f32":
        e.valu(f"v_mov_b32_e32 v{p.tscale}, {LOG2E}", [p.tscale])
    if not p.scaled:
        # ---- maxima of the seeded integer scores ---------------------------------------------------
        for rb in range(p.rb):
            e.need_mfma_result(p.S[rb])
            evens = [p.S[rb] + i for i in range(16) if not i & 2]
            odds = [p.S[rb] + i for i in range(16) if i & 2]
            for target, registers in ((p.mx0, evens), (p.mx1, odds)):
                if rb == 0:
                    e.valu(f"v_max_i32_e32 v{target}, v{registers[0]}, v{registers[1]}", [target])
                    registers = registers[2:]
                while registers:
                    e.valu(f"v_max3_i32 v{target}, v{target}, v{registers[0]}, v{registers[1]}", [target])
                    registers = registers[2:]
        e.valu(f"v_sub_f32_e32 v{p.mx0}, v{p.mx0}, v{p.seedval}", [p.mx0])
        e.valu(f"v_sub_f32_e32 v{p.mx1}, v{p.mx1}, v{p.seedval}", [p.mx1])
        e.valu(f"v_mov_b32_e32 v{p.negm}, {MINUS_U8_OFFSET}", [p.negm])
        e.valu(f"v_fma_f32 v{p.mx0}, v{p.mx0}, v{p.sc0}, v{p.negm}", [p.mx0])
        e.valu(f"v_fma_f32 v{p.mx1}, v{p.mx1}, v{p.sc1}, v{p.negm}", [p.mx1])
        e.valu(f"v_max_f32_e32 v{p.mx0}, v{p.mx0}, v{p.mx1}", [p.mx0])
    else:
        # ---- scaled scores and their maximum -------------------------------------------------------
        if p.mask == "bias":
            e.wait_lds(p.PK[0])
            probe = p.PK[0]
            e.valu(f"v_or3_b32 v{probe}, v{probe}, v{probe + 1}, v{probe + 2}", [probe])
            e.valu(f"v_or_b32_e32 v{probe}, v{probe}, v{probe + 3}", [probe])
            e.valu(f"v_lshlrev_b32_e32 v{probe}, 1, v{probe}", [probe])  # (a zero of either sign)
            e.valu(f"v_cmp_ne_u32_e32 vcc, 0, v{probe}")
        if p.mask == "lanes":
            e.valu(f"v_mov_b32_e32 v{p.tscale}, {NEG_INF}", [p.tscale])
        for rb in range(p.rb):
            e.need_mfma_result(p.S[rb])
            block = [p.S[rb] + i for i in range(16)]
            for register in block:
                e.valu(f"v_sub_f32_e32 v{register}, v{register}, v{p.seedval}", [register])
            for i, register in enumerate(block):
                e.valu(f"v_mul_f32_e32 v{register}, v{register}, v{scale_of(i)}", [register])
            if p.mask == "f32":
                # A term of -inf leaves -inf, one that is no number a score the maximum does not see
                # and whose probability is zero: both as if the key were hidden.  Terms of +inf hide
                # their keys too; they show in the maximum below.
                for first in range(0, 16, 4):
                    for r in range(4):
                        e.valu(f"v_mul_f32_e32 v{p.T[r]}, v{p.M + rb * 16 + first + r}, v{p.tscale}", [p.T[r]])
                    for r in range(4):
                        register = block[first + r]
                        e.valu(f"v_add_f32_e32 v{register}, v{register}, v{p.T[r]}", [register])
            if p.mask == "lanes":
                if rb == 1:
                    e.ins("s_waitcnt lgkmcnt(0)")
                    e.lds_queue = []
                for i, register in enumerate(block):
                    e.valu(f"v_cndmask_b32_e64 v{register}, v{p.tscale}, v{register}, {pair(p.words + 2 * i)}", [register])
                if rb == 0:  # the words of the second key block over those of the first
                    e.ins(f"s_load_dwordx16 s[{p.words}:{p.words + 15}], {pair(p.words_at)}, 0x80")
                    e.ins(f"s_load_dwordx16 s[{p.words + 16}:{p.words + 31}], {pair(p.words_at)}, 0xc0")
        if p.mask == "bias":
            e.ins(f"s_cbranch_vccz {label}_zerorow")
            # (the V fragment and probability registers are free: the terms of one key block at a time)
            terms = p.VF[0] if p.cb == 2 else p.PK[0] - 16
            assert p.PK[1] + 4 >= terms + 16
            for rb in range(p.rb):
                for b4 in range(4):
                    e.ins(f"ds_read_b128 v[{terms + b4 * 4}:{terms + b4 * 4 + 3}], v{p.seedaddr} "
                          f"offset:{base + p.bias_region - SEED_BIAS + rb * 128 + b4 * 32}")
                e.ins("s_waitcnt lgkmcnt(0)")
                for i in range(16):
                    register = p.S[rb] + i
                    e.valu(f"v_add_f32_e32 v{register}, v{register}, v{terms + i}", [register])
            e.raw(f"{label}_zerorow:")
        def row_maximum():
            e.valu(f"v_mov_b32_e32 v{p.mx0}, {ROW_FLOOR}", [p.mx0])
            e.valu(f"v_max_f32_e32 v{p.mx1}, v{scores[0]}, v{scores[1]}", [p.mx1])
            for index, at in enumerate(range(2, len(scores), 2)):
                target = p.mx1 if index & 1 else p.mx0
                e.valu(f"v_max3_f32 v{target}, v{target}, v{scores[at]}, v{scores[at + 1]}", [target])
            e.valu(f"v_max_f32_e32 v{p.mx0}, v{p.mx0}, v{p.mx1}", [p.mx0])

        row_maximum()
        if p.mask == "f32":
            # some score is +inf: take the keys out whose term is no finite number
            e.valu(f"v_cmp_eq_f32_e32 vcc, {POS_INF}, v{p.mx0}")
            e.nop(4)
            e.ins(f"s_cbranch_vccz {label}_finite")
            e.valu(f"v_mov_b32_e32 v{p.rowsum}, {NEG_INF}", [p.rowsum])
            for group in range(8):
                for r in range(4):
                    e.ins(f"v_cmp_class_f32_e64 {pair(p.pairs[r])}, v{p.M + group * 4 + r}, s{p.klass}")
                for r in range(4):
                    register = scores[group * 4 + r]
                    e.valu(f"v_cndmask_b32_e64 v{register}, v{p.rowsum}, v{register}, {pair(p.pairs[r])}", [register])
            row_maximum()
            e.raw(f"{label}_finite:")
        e.valu(f"v_add_f32_e32 v{p.mx0}, {MINUS_U8_OFFSET}, v{p.mx0}", [p.mx0])
    e.valu(f"v_mov_b32_e32 v{p.mx1}, v{p.mx0}", [p.mx1])
    e.nop(2)
    e.valu(f"v_permlane32_swap_b32_e32 v{p.mx0}, v{p.mx1}", [p.mx0, p.mx1])  # the other half's maximum
    e.nop(2)
    e.valu(f"v_max_f32_e32 v{p.mx0}, v{p.mx0}, v{p.mx1}", [p.mx0])  # tile maximum - 7.99 of the row
    # ---- online-softmax state: the reference only moves when a tile maximum exceeds it by more than 8
    e.valu(f"v_add_f32_e32 v{p.tmp}, 0x41000000, v{p.mrun}", [p.tmp])
    e.valu(f"v_cmp_gt_f32_e32 vcc, v{p.mx0}, v{p.tmp}")
    # ---- V fragments of key block 0 (their latency hides behind the scaling pass) --------------------
    for cb in range(p.cb):
        e.ds_read(p.VF[cb], p.VA[0], p.v_region(stage) + cb * 32 * p.keys)
    e.nop(4)
    e.ins(f"s_cbranch_vccz {label}_keep")
    e.valu(f"v_sub_f32_e32 v{p.tmp}, v{p.mrun}, v{p.mx0}", [p.tmp])
    e.valu(f"v_exp_f32_e32 v{p.tmp}, v{p.tmp}", [p.tmp], trans=True)
    e.nop(1)
    e.valu(f"v_cndmask_b32_e32 v{p.tmp}, 1.0, v{p.tmp}, vcc", [p.tmp])
    e.valu(f"v_cndmask_b32_e32 v{p.mrun}, v{p.mrun}, v{p.mx0}, vcc", [p.mrun])
    e.valu(f"v_mul_f32_e32 v{p.dpart}, v{p.dpart}, v{p.tmp}", [p.dpart])
    for cb in range(p.cb):
        for i in range(16):
            e.valu(f"v_mul_f32_e32 v{p.O[cb] + i}, v{p.O[cb] + i}, v{p.tmp}", [p.O[cb] + i])
    e.raw(f"{label}_keep:")
    e.valu(f"v_sub_f32_e32 v{p.tscale}, v{p.mx0}, v{p.mrun}", [p.tscale])
    e.valu(f"v_exp_f32_e32 v{p.tscale}, v{p.tscale}", [p.tscale], trans=True)

    # ---- exponent arguments in place of the scores -----------------------------------------------------
    if p.scaled:
        for register in scores:
            e.valu(f"v_sub_f32_e32 v{register}, v{register}, v{p.mx0}", [register])
    else:
        e.valu(f"v_sub_f32_e32 v{p.negm}, 0, v{p.mx0}", [p.negm])
        for rb in range(p.rb):
            for i in range(16):
                register = p.S[rb] + i
                e.valu(f"v_sub_f32_e32 v{register}, v{register}, v{p.seedval}", [register])
            for i in range(16):
                register = p.S[rb] + i
                e.valu(f"v_fma_f32 v{register}, v{register}, v{scale_of(i)}, v{p.negm}", [register])
    e.valu(f"v_mov_b32_e32 v{p.rowsum}, 0", [p.rowsum])

    def pack_group(rb, b4, pk):
        """Four scores -> one register of signed probability bytes, and their sum."""
        registers = [p.S[rb] + b4 * 4 + r for r in range(4)]
        # (tight: over scores of this group or of one already packed)
        targets = registers if p.tight else p.T
        for r in range(4):
            e.valu(f"v_exp_f32_e32 v{targets[r]}, v{registers[r]}", [targets[r]], trans=True)
        for r in range(4):
            e.need_trans(targets[r])
            previous = "0" if r == 0 else f"v{pk + b4}"
            e.valu(f"v_cvt_pk_u8_f32 v{pk + b4}, v{targets[r]}, {r}, {previous}", [pk + b4])
        e.valu(f"v_sad_u8 v{p.rowsum}, v{pk + b4}, 0, v{p.rowsum}", [p.rowsum])
        e.valu(f"v_xor_b32_e32 v{pk + b4}, 0x80808080, v{pk + b4}", [pk + b4])

    def value_products(cb, pk):
        for b4 in range(4):
            e.wait_lds(p.ACC[cb] + b4 * 4)
        e.wait_lds(p.VF[cb])
        e.mfma(p.ACC[cb], p.VF[cb], pk, p.ACC[cb])

    e.ins(f"s_setprio {prio[2]}")
    for b4 in range(4):
        pack_group(0, b4, p.PK[0])
    for rb in range(1, p.rb):
        previous, current = p.PK[(rb - 1) & 1], p.PK[rb & 1]
        for b4 in range(4):
            if b4 % (4 // p.cb) == 0:
                cb = b4 // (4 // p.cb)
                value_products(cb, previous)
                e.ds_read(p.VF[cb], p.VA[rb], p.v_region(stage) + cb * 32 * p.keys)
            pack_group(rb, b4, current)
    for cb in range(p.cb):
        value_products(cb, p.PK[(p.rb - 1) & 1])
    total = p.rowsum if p.tight else p.T[0]
    e.valu(f"v_cvt_f32_u32_e32 v{total}, v{p.rowsum}", [total])
    e.valu(f"v_fmac_f32_e32 v{p.dpart}, v{total}, v{p.tscale}", [p.dpart])
    # ---- scalar loads of the next tile: waited for at the next barrier ------------------------------
    if p.listed:
        e.ins(f"s_lshl_b32 s{p.tmp_s}, s{p.tnext}, 4")
        e.ins(f"s_add_u32 s{p.tmp_s}, s{p.ksptr}, s{p.tmp_s}")
        e.ins(f"s_addc_u32 s{p.tmp_s + 1}, s{p.ksptr + 1}, 0")
        e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.tmp_s)}, 0x0")
        if p.mask == "lanes":
            load_words(e, p, p.tnext)
        e.ins(f"s_add_u32 s{p.index}, s{p.index}, 1")
        e.ins(f"s_min_u32 s{p.index}, s{p.index}, s{p.last}")
        e.ins(f"s_lshl_b32 s{p.tmp_s}, s{p.index}, 2")
        e.ins(f"s_add_u32 s{p.tmp_s}, s{p.list}, s{p.tmp_s}")
        e.ins(f"s_addc_u32 s{p.tmp_s + 1}, s{p.list + 1}, 0")
        e.ins(f"s_load_dword s{p.tafter}, {pair(p.tmp_s)}, 0x0")
    else:
        add64(e, p.ksptr, 16)
        e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.ksptr)}, 0x0")
    # ---- output update -------------------------------------------------------------------------------
    e.ins(f"s_setprio {prio[3]}")
    for cb in range(p.cb):
        e.need_mfma_result(p.ACC[cb])
        for i in range(0, 16, 4):
            targets = [p.ACC[cb] + i + j for j in range(4)] if p.tight else p.T
            for j in range(4):
                e.valu(f"v_sub_f32_e32 v{targets[j]}, v{p.ACC[cb] + i + j}, v{p.seedval}", [targets[j]])
            for j in range(4):
                e.valu(f"v_fmac_f32_e32 v{p.O[cb] + i + j}, v{targets[j]}, v{p.tscale}", [p.O[cb] + i + j])


def generate(p, prio):
    e = Emitter()
    e.comment("set-up: operands into fixed scalar registers")
    for target, name in ((p.kptr, "kptr"), (p.vptr, "vptr"), (p.sumptr, "sumptr"), (p.ksptr, "ksptr")):
        e.ins(f"s_mov_b64 {pair(target)}, %[{name}]")
    e.ins(f"s_mov_b32 s{p.count}, %[count]")
    e.ins(f"s_mov_b32 s{p.qs2}, %[qs2]")
    e.ins(f"s_mul_i32 s{p.vstep}, %[padded], {p.v_rows}")
    if p.listed:
        e.ins(f"s_mov_b64 {pair(p.list)}, %[list]")
    if p.mask is not None:
        e.ins(f"s_mov_b64 {pair(p.maskptr)}, %[mask]")
    # LDS base: lane 0 of the seed address register holds base + SEED_BIAS
    e.ins(f"v_readfirstlane_b32 s{p.lds}, v{p.seedaddr}")
    e.ins(f"s_sub_u32 s{p.lds}, s{p.lds}, {SEED_BIAS}")
    e.ins(f"s_mov_b32 s{p.halfmask}, 0")
    e.ins(f"s_mov_b32 s{p.halfmask + 1}, -1")
    # this wave's copy slots (the V slots are one tile behind the K slots) and its share of the sources
    e.ins(f"s_mul_i32 s{p.tmp_s}, %[wave], {p.copies * 1024}")
    e.ins(f"s_add_u32 s{p.klds}, s{p.lds}, s{p.tmp_s}")
    e.ins(f"s_add_u32 s{p.kptr}, s{p.kptr}, s{p.tmp_s}")
    e.ins(f"s_addc_u32 s{p.kptr + 1}, s{p.kptr + 1}, 0")
    e.ins(f"s_mul_i32 s{p.tmp_s}, %[wave], {p.copies}")
    e.ins(f"s_mul_hi_u32 s{p.tmp2_s}, s{p.tmp_s}, s{p.vstep}")
    e.ins(f"s_mul_i32 s{p.tmp_s}, s{p.tmp_s}, s{p.vstep}")
    e.ins(f"s_add_u32 s{p.vptr}, s{p.vptr}, s{p.tmp_s}")
    e.ins(f"s_addc_u32 s{p.vptr + 1}, s{p.vptr + 1}, s{p.tmp2_s}")
    if p.mask == "f32":
        e.ins(f"s_mov_b32 s{p.mstep}, %[maskstep]")
        e.ins(f"s_movk_i32 s{p.klass}, 0x1f8")  # finite numbers
        e.ins(f"s_lshl_b32 s{p.tmp_s}, %[wave], 13")
        e.ins(f"s_add_u32 s{p.mlds}, s{p.lds}, s{p.tmp_s}")
        e.ins(f"s_add_u32 s{p.mlds}, s{p.mlds}, {p.mask_region}")
    if p.listed:
        # list[0] is the tile whose copies are in flight, list[1] the first one this loop copies
        e.ins(f"s_load_dwordx2 {pair(p.tmp_s)}, {pair(p.list)}, 0x0")
        e.ins(f"s_mov_b32 s{p.last}, s{p.count}")  # the loop reads no entry behind the tile it copies last
        e.ins(f"s_mov_b32 s{p.index}, 1")
        e.ins("s_waitcnt lgkmcnt(0)")
        e.ins(f"s_mov_b32 s{p.tafter}, s{p.tmp_s + 1}")
        e.ins(f"s_mov_b32 s{p.tnext}, s{p.tmp_s}")
        e.ins(f"s_lshl_b32 s{p.tmp_s}, s{p.tnext}, 4")
        e.ins(f"s_add_u32 s{p.tmp_s}, s{p.ksptr}, s{p.tmp_s}")
        e.ins(f"s_addc_u32 s{p.tmp_s + 1}, s{p.ksptr + 1}, 0")
        e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.tmp_s)}, 0x0")
        if p.mask == "lanes":
            load_words(e, p, p.tnext)
    else:
        e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.ksptr)}, 0x0")
    e.ins(f"v_mov_b32_e32 v{p.seedval}, 0x4b400000")
    if p.seeds_kept:
        for r in range(16):
            e.valu(f"v_mov_b32_e32 v{p.SEEDS + r}, v{p.seedval}", [p.SEEDS + r])
    e.raw("Lrisa_loop_%=:")
    tile_body(e, p, 0, prio, "Lrisa_a_%=")
    e.ins(f"s_sub_u32 s{p.count}, s{p.count}, 1")
    e.ins(f"s_cmp_eq_u32 s{p.count}, 0")
    e.ins("s_cbranch_scc1 Lrisa_done_%=")
    tile_body(e, p, 1, prio, "Lrisa_b_%=")
    e.ins(f"s_sub_u32 s{p.count}, s{p.count}, 1")
    e.ins(f"s_cmp_lg_u32 s{p.count}, 0")
    e.ins("s_cbranch_scc1 Lrisa_loop_%=")
    e.raw("Lrisa_done_%=:")
    e.ins("s_waitcnt lgkmcnt(0)")
    e.ins("s_setprio 0")
    return e


PROGRAMS = (
    Program("scaled_d128k128", 128, 128, scaled=True),
    Program("raw_d128k64", 128, 64, scaled=False),
    Program("f32mask_d128k64", 128, 64, scaled=True, mask="f32"),
    Program("bias_d128k128", 128, 128, scaled=True, mask="bias"),
    Program("bias_listed_d128k128", 128, 128, scaled=True, mask="bias", listed=True),
    Program("lanes_listed_d128k64", 128, 64, scaled=True, mask="lanes", listed=True),
    Program("raw_d64k64", 64, 64, scaled=False),
    Program("scaled_d64k64", 64, 64, scaled=True),
    Program("bias_d64k64", 64, 64, scaled=True, mask="bias"),
    Program("bias_listed_d64k64", 64, 64, scaled=True, mask="bias", listed=True),
    Program("lanes_listed_d64k64", 64, 64, scaled=True, mask="lanes", listed=True, tight=True),
)


def operands(p):
    """(outputs, inputs) as (constraint, C++ expression) pairs."""
    block = lambda first, count: f"{{v[{first}:{first + count - 1}]}}" if count > 1 else f"{{v{first}}}"
    outputs = [(block(p.O[cb], 16), f"out{cb}") for cb in range(p.cb)]
    outputs += [(block(p.mrun, 1), "m_run"), (block(p.dpart, 1), "d_part")]
    inputs = [(block(p.Q[kk], 4), f"qreg[{kk}]") for kk in range(p.kk)] + [(block(p.qscale, 1), "q_scale")]
    if p.ka is not None:
        inputs.append((block(p.ka, 1), "k_address[0]"))
    else:
        inputs += [(block(register, 1), f"k_address[{kk}]") for kk, register in enumerate(p.KA)]
    if not p.va_shared:
        inputs += [(block(register, 1), f"v_address[{rb}]") for rb, register in enumerate(p.VA)]
    inputs.append((block(p.seedaddr, 1), "seed_address"))
    inputs += [(block(register, 1), f"k_share[{i}]") for i, register in enumerate(p.KC)]
    inputs += [(block(register, 1), f"v_share[{i}]") for i, register in enumerate(p.VC)]
    if p.mask == "f32":
        inputs += [(block(p.maddr, 1), "mask_address"), (block(p.mch, 1), "mask_chunk"), (block(p.mrow, 1), "mask_row_share")]
    named = [("kptr", "k_source"), ("vptr", "v_source"), ("sumptr", "sum_source"), ("ksptr", "ks_source"),
             ("count", "walk"), ("wave", "wave"), ("qs2", "qs2"), ("padded", "p.padded")]
    if p.listed:
        named.append(("list", "list"))
    if p.mask is not None:
        named.append(("mask", "mask_source"))
    if p.mask == "f32":
        named.append(("maskstep", "mask_step"))
    return outputs, inputs, named


def render(p, prio=(0, 1, 2, 0)):
    """The asm statement as the include file holds it."""
    e = generate(p, prio)
    outputs, inputs, named = operands(p)
    text = "asm volatile(RISA_LOOP_AT_EVEN_WORD\n" + "".join('"{}\\n\\t"\n'.format(line.replace('"', '\\"')) for line in e.lines)
    text += "    : " + ", ".join(f'"+{c}"({x})' for c, x in outputs) + "\n"
    text += "    : " + ", ".join(f'"{c}"({x})' for c, x in inputs) + ",\n"
    text += "      " + ", ".join(f'[{n}] "s"({x})' for n, x in named) + "\n"
    pinned = set()
    for constraint, _ in outputs + inputs:
        numbers = [int(t) for t in constraint.strip("{}").replace("v", "").replace("[", "").replace("]", "").split(":")]
        pinned |= set(range(numbers[0], numbers[-1] + 1))
    clobbered = [f"v{r}" for r in range(p.next_vgpr) if r not in pinned]
    clobbered += [f"s{r}" for r in range(FIRST_SGPR, p.next_sgpr)] + ["vcc", "scc", "m0", "memory"]
    text += "    : " + ", ".join(f'"{name}"' for name in clobbered) + ");\n"
    return text


def main():
    parser = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    parser.add_argument("--outdir", type=pathlib.Path, default=pathlib.Path(__file__).resolve().parent)
    args = parser.parse_args()
    for program in PROGRAMS:
        (args.outdir / f"tile_loop_{program.name}.inc").write_text(render(program))


if __name__ == "__main__":
    main()
