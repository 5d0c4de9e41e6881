#!/usr/bin/env python3
"""Writes the tile walks of head dim 256 with thirty-two queries per wavefront (128-key tiles), one
`asm volatile` statement per program, as d256_loop_<name>.inc beside this file.

    python3 gen_d256_loops.py

A program walks every listed tile of a query block, the last one included: output accumulators (128
registers), scores (64) and Q (32) leave 31 registers for everything else, which the compiler cannot
schedule without spilling (380 registers, one wavefront per SIMD).

The arithmetic of a score is the C++ kernels' (attention_kernel.hpp, attention_narrow_kernel.hpp), in
the order of gen_dense_loop.py and gen_tile_loops.py.  What differs is the staging.  A K and a V tile are 64
KB, so two workgroups per compute unit leave no room for two stages.  K of the next tile is copied
behind the barrier at which every wavefront has left the score product, V of a tile behind the one at
which every wavefront has left the value product before it:

    barrier A   K of this tile landed; V of the tile before is free   -> copy V of this tile
    score product, maxima, exponent arguments
    barrier B   V of this tile landed; K of this tile is free         -> copy K of the next tile
    exponentials, value product, output update

Modes:  raw, scaled, bias (additive row of a key-only mask), bias_listed (over a tile list), as in
gen_tile_loops.py.  The last tile hides the keys past the end and, under the causal rule, past the query.
"""
import argparse
import pathlib
import sys

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent))
from gen_dense_loop import Emitter, add64  # noqa: E402
from gen_tile_loops import MINUS_U8_OFFSET, NEG_INF, ROW_FLOOR, pair  # noqa: E402

FIRST_SGPR = 36
DIM, KEYS, KK, CB, RB, COPIES = 256, 128, 8, 8, 4, 8
TILE_BYTES = DIM * KEYS
# LDS: accumulator seeds, additive row, (channel scale and centre of the epilogue,) K tile, V tile
SEED_REGION, BIAS_REGION, K_REGION, V_REGION = 0, 1024, 4096, 4096 + TILE_BYTES
PAST_END = "0xf149f2ca"  # -1e30: a negative integer, so it never wins the integer maximum

# ---- vector registers ---------------------------------------------------------------------------
O = [16 * cb for cb in range(CB)]
S = [128 + 16 * rb for rb in range(RB)]
Q = [192 + 4 * kk for kk in range(KK)]
X = 224                 # score seeds, K fragments, softmax temporaries, terms of the additive row, V fragments
F = 240                 # one more fragment; row sum
MRUN, DPART, QSCALE, SEEDVAL, KA, VA, VC, KC = range(244, 252)
SC0, SC1, TSCALE = 252, 253, 254   # (K fragment addresses in the score product)
PK = S[0]               # probabilities of key block rb in PK + 4 * rb, over scores already packed
ACC = [X, S[2], S[3]]    # accumulators of the value product
VF = [S[1] + 4 * rb for rb in range(4)]  # and its V fragments
# Vector work beside the second half of the score product: from its fourth product on, five
# instructions behind each.
PAUSE, BESIDE = 3, 5
# Wave priorities of the score product, the maxima, the exponentials and the value product.  16/4 heads
# x 8192, whole call, plain / causal: 0 1 2 0 (the loops of head dim 128) 654 / 380 us, all 0 659 / 372,
# 1 1 1 0 647 / 372, 1 0 2 0 654 / 382, 2 1 3 0 639 / 362.
PRIORITIES = (2, 1, 3, 0)
LAST_VGPR = 254


class Program:
    def __init__(self, name, scaled, bias=False, listed=False):
        self.name, self.scaled, self.bias, self.listed = name, scaled, bias, listed
        self.next_sgpr = FIRST_SGPR
        stake = self.stake
        self.ks = stake(4, 4)
        self.kptr, self.vptr, self.sumptr, self.ksptr = stake(2), stake(2), stake(2), stake(2)
        self.kat, self.at = stake(2), stake(2)
        self.halfmask = stake(2)
        self.list, self.maskptr = stake(2), stake(2)
        self.count, self.klds, self.qs2, self.vstep, self.wave = stake(1), stake(1), stake(1), stake(1), stake(1)
        self.tile, self.tnext, self.tafter, self.index, self.last = stake(1), stake(1), stake(1), stake(1), stake(1)
        self.rem, self.remq = stake(1), stake(1)
        assert self.next_sgpr <= 100

    def stake(self, count, align=None):
        align = align or count
        self.next_sgpr = -(-self.next_sgpr // align) * align
        first = self.next_sgpr
        self.next_sgpr += count
        return first


def address(e, p, target, pointer, tile, bits):
    """Scalar pair `target`: pointer + (tile << bits) of a listed tile."""
    e.ins(f"s_lshl_b32 s{target}, s{tile}, {bits}")
    e.ins(f"s_add_u32 s{target}, s{pointer}, s{target}")
    e.ins(f"s_addc_u32 s{target + 1}, s{pointer + 1}, 0")


def lane_times_16(e, register):
    e.ins(f"v_mbcnt_lo_u32_b32 v{register}, -1, 0")
    e.ins(f"v_mbcnt_hi_u32_b32 v{register}, -1, v{register}")
    e.ins(f"v_lshlrev_b32_e32 v{register}, 4, v{register}")


def k_copies(e, p, label, lane16):
    """K (and the additive row) of the next tile, as a list of pieces to spread over other work.  The
    lane share of copy i is KC ^ (i % 4) * 64 (the swizzle's period), so copies of one share go together."""
    def start():
        if p.listed:
            address(e, p, p.kat, p.kptr, p.tnext, 15)
        else:
            e.ins(f"s_mov_b64 {pair(p.kat)}, {pair(p.kptr)}")

    def copy(i, first):
        def emit():
            if first:
                start()
            e.ins(f"s_add_u32 s{p.at}, s{p.kat}, {i * 1024}")
            e.ins(f"s_addc_u32 s{p.at + 1}, s{p.kat + 1}, 0")
            e.ins(f"s_add_u32 m0, s{p.klds}, {K_REGION + i * 1024}")
            e.ins("s_nop 0")
            e.ins(f"global_load_lds_dwordx4 v{KC}, {pair(p.at)}")
            if i >= 4:
                e.valu(f"v_xor_b32_e32 v{KC}, {64 if i % 2 == 0 else 192}, v{KC}", [KC])
        return emit

    def bias_copy():
        e.ins(f"s_cmp_lg_u32 s{p.wave}, 1")
        e.ins(f"s_cbranch_scc1 {label}_nobias")
        if p.listed:
            address(e, p, p.at, p.maskptr, p.tnext, 9)
        else:
            e.ins(f"s_mov_b64 {pair(p.at)}, {pair(p.maskptr)}")
        lane_times_16(e, lane16)
        e.ins("s_mov_b64 exec, 0xffffffff")
        e.ins(f"s_mov_b32 m0, {BIAS_REGION}")
        e.ins("s_nop 0")
        e.ins(f"global_load_lds_dwordx4 v{lane16}, {pair(p.at)}")
        e.ins("s_mov_b64 exec, -1")
        e.raw(f"{label}_nobias:")

    pieces = [copy(i, at == 0) for at, i in enumerate((0, 4, 1, 5, 2, 6, 3, 7))]
    if p.bias:
        pieces.append(bias_copy)
    return pieces


def v_copies(e, p, label):
    """V and the accumulator seeds of this tile; odd copies use VC ^ 64."""
    def copy(at, i):
        def emit():
            if at == 0:
                if p.listed:
                    address(e, p, p.at, p.vptr, p.tile, 7)
                else:
                    e.ins(f"s_mov_b64 {pair(p.at)}, {pair(p.vptr)}")
                e.ins(f"s_mov_b64 {pair(p.kat)}, {pair(p.at)}")
            elif i == 1:
                e.ins(f"s_add_u32 s{p.at}, s{p.kat}, s{p.vstep}")
                e.ins(f"s_addc_u32 s{p.at + 1}, s{p.kat + 1}, 0")
                e.valu(f"v_xor_b32_e32 v{VC}, 64, v{VC}", [VC])
            else:
                for _ in range(2):
                    e.ins(f"s_add_u32 s{p.at}, s{p.at}, s{p.vstep}")
                    e.ins(f"s_addc_u32 s{p.at + 1}, s{p.at + 1}, 0")
            e.ins(f"s_add_u32 m0, s{p.klds}, {V_REGION + i * 1024}")
            e.ins("s_nop 0")
            e.ins(f"global_load_lds_dwordx4 v{VC}, {pair(p.at)}")
            if i == 7:
                e.valu(f"v_xor_b32_e32 v{VC}, 64, v{VC}", [VC])
        return emit
    return [copy(at, i) for at, i in enumerate((0, 2, 4, 6, 1, 3, 5, 7))]


def seed_copy(e, p, label, lane16):
    e.ins(f"s_cmp_lg_u32 s{p.wave}, 0")
    e.ins(f"s_cbranch_scc1 {label}_noseed")
    if p.listed:
        address(e, p, p.at, p.sumptr, p.tile, 10)
    else:
        e.ins(f"s_mov_b64 {pair(p.at)}, {pair(p.sumptr)}")
    lane_times_16(e, lane16)
    e.ins(f"s_mov_b32 m0, {SEED_REGION}")
    e.ins("s_nop 0")
    e.ins(f"global_load_lds_dwordx4 v{lane16}, {pair(p.at)}")
    e.raw(f"{label}_noseed:")


def tile_body(e, p, last, prio, label):
    e.comment(f"===== {'last tile' if last else 'tile'} =====")
    for r in range(16):
        e.valu(f"v_mov_b32_e32 v{X + r}, v{SEEDVAL}", [X + r])
    e.ins("s_waitcnt vmcnt(0) lgkmcnt(0)")
    e.ins("s_barrier")  # A
    e.ins(f"s_setprio {prio[0]}")
    e.lds_queue = []
    if p.listed:
        e.ins(f"s_mov_b32 s{p.tile}, s{p.tnext}")
        e.ins(f"s_mov_b32 s{p.tnext}, s{p.tafter}")

    # ---- S^T = K Q^T -----------------------------------------------------------------------------
    # First k-step of all four key blocks (its fragments stand in the last block's registers, the seeds
    # are free behind it), the other steps of blocks 0 and 1, then those of 2 and 3: beside these the
    # scores of the first two lose their seed and enter the maxima.
    order = [(0, rb) for rb in range(RB)] + [(kk, rb) for half in (0, 2) for kk in range(1, KK) for rb in (half, half + 1)]
    free, slot, next_read, addressed = [], {}, 0, 0

    def read_fragment(at):
        nonlocal next_read, addressed
        kk, rb = order[next_read]
        if kk != addressed:
            e.valu(f"v_xor_b32_e32 v{SC0}, {kk * 32}, v{KA}", [SC0])
            addressed = kk
        slot[kk, rb] = at
        e.ds_read(at, SC0 if kk else KA, rb * 32 * DIM)
        next_read += 1

    mx0, mx1, negm, tmp, upper0, upper1, rem, past = (X + i for i in range(8))
    early0, early1 = TSCALE, SC1  # maxima while the registers above hold fragments

    def unseed(rb):
        return [lambda r=S[rb] + i: e.valu(f"v_sub_f32_e32 v{r}, v{r}, v{SEEDVAL}", [r]) for i in range(16)]

    def maxima(rb, targets, sources):
        """The block's two scale groups into `targets`; `sources` hold the maxima so far."""
        steps = []
        for target, source, group in zip(targets, sources, (0, 2)):
            registers = [S[rb] + i for i in range(16) if i & 2 == group]
            if source is None:
                steps.append(lambda t=target, a=registers[0], c=registers[1]: e.valu(f"v_max_f32_e32 v{t}, v{a}, v{c}", [t]))
                registers, source = registers[2:], target
            for at in range(0, len(registers), 2):
                steps.append(lambda t=target, o=source, a=registers[at], c=registers[at + 1]:
                             e.valu(f"v_max3_f32 v{t}, v{o}, v{a}, v{c}", [t]))
                source = target
        return steps

    with_maxima = not p.scaled and not last
    beside = []
    for rb in (0, 1):
        beside.append(lambda rb=rb: e.need_mfma_result(S[rb]))
        beside += unseed(rb)
        if with_maxima:
            beside += maxima(rb, (early0, early1), (None, None) if rb == 0 else (early0, early1))

    for at in (S[3], S[3] + 4, S[3] + 8, F):
        read_fragment(at)
    seed_copy(e, p, label, TSCALE)
    copies = v_copies(e, p, label)
    for at_product, (kk, rb) in enumerate(order):
        at = slot[kk, rb]
        e.wait_lds(at)
        if kk == 0:
            e.need_valu_result_for_mfma(range(X, X + 16))
        e.mfma(S[rb], at, Q[kk], X if kk == 0 else S[rb])
        if kk == 0 and rb < 3:
            continue
        free.append(at)
        if kk == 0:
            free += [X, X + 4, X + 8, X + 12]
        while free and next_read < len(order):
            read_fragment(free.pop(0))
        if copies and kk > 0:
            copies.pop(0)()
        if at_product >= 18 + PAUSE:
            for _ in range(BESIDE):
                if beside:
                    beside.pop(0)()
    for step in beside:
        step()
    if not p.listed:
        if not last:
            add64(e, p.vptr, KEYS)
            add64(e, p.sumptr, DIM * 4)

    e.ins(f"s_setprio {prio[1]}")

    def score_scales():
        # K scales -> score scales of this lane's two key groups
        if p.bias:
            # the row of additive terms, 16 bytes per lane: is any of them not zero?
            lane_times_16(e, tmp)
            e.valu(f"v_and_b32_e32 v{tmp}, {KEYS * 4 - 1}, v{tmp}", [tmp])
            e.ds_read(F, tmp, BIAS_REGION)
        for register, at in ((upper0, 2), (upper1, 3), (SC0, 0), (SC1, 1)):
            e.valu(f"v_mov_b32_e32 v{register}, s{p.ks + at}", [register])
        for register, upper in ((SC0, upper0), (SC1, upper1)):
            e.valu(f"v_cndmask_b32_e64 v{register}, v{register}, v{upper}, {pair(p.halfmask)}", [register])
        for register in (SC0, SC1):
            e.valu(f"v_mul_f32_e32 v{register}, v{QSCALE}, v{register}", [register])
        for register in (SC0, SC1):
            e.valu(f"v_mul_f32_e32 v{register}, s{p.qs2}, v{register}", [register])
    scores = [S[rb] + i for rb in range(RB) for i in range(16)]
    scale_of = lambda i: SC1 if i & 2 else SC0

    def hide(bits):
        """Last tile: keys past the end (and past the query) out of the scores."""
        e.ins(f"s_min_u32 s{p.at}, s{p.rem}, s{p.remq}")
        e.ins(f"s_cmp_ge_u32 s{p.at}, {KEYS}")
        e.ins(f"s_cbranch_scc1 {label}_whole")
        # rem = min(keys left, keys up to the query) - 4 * half: this lane keeps its keys below
        e.ins(f"v_mbcnt_lo_u32_b32 v{rem}, -1, 0")
        e.ins(f"v_mbcnt_hi_u32_b32 v{rem}, -1, v{rem}")
        e.valu(f"v_lshrrev_b32_e32 v{past}, 5, v{rem}", [past])
        e.valu(f"v_and_b32_e32 v{rem}, 31, v{rem}", [rem])
        e.valu(f"v_add_u32_e32 v{rem}, s{p.remq}, v{rem}", [rem])
        e.valu(f"v_min_i32_e32 v{rem}, s{p.rem}, v{rem}", [rem])
        e.valu(f"v_lshlrev_b32_e32 v{past}, 2, v{past}", [past])
        e.valu(f"v_sub_u32_e32 v{rem}, v{rem}, v{past}", [rem])
        e.valu(f"v_mov_b32_e32 v{past}, {bits}", [past])
        # A select reads its comparison two wait states behind it (nothing in hardware holds it back), so
        # three scalar pairs take turns.  (Keys below 64 are inline constants, which is what a comparison
        # into such a pair takes.)
        masks = ["vcc", pair(p.kat), pair(p.at)]
        selects = []
        for rb in range(RB):
            if rb == 2:
                e.valu(f"v_add_u32_e32 v{rem}, 0xffffffc0, v{rem}", [rem])  # - 64
            for i in range(16):
                mask = masks[(rb * 16 + i) % 3]
                e.valu(f"v_cmp_lt_i32_e64 {mask}, {rb % 2 * 32 + (i >> 2) * 8 + (i & 3)}, v{rem}")
                selects.append(lambda r=S[rb] + i, m=mask: e.valu(f"v_cndmask_b32_e64 v{r}, v{past}, v{r}, {m}", [r]))
                if len(selects) > 2:
                    selects.pop(0)()
        for select in selects:
            select()
        e.raw(f"{label}_whole:")

    for rb in (2, 3):
        e.need_mfma_result(S[rb])
        for step in unseed(rb):
            step()
    if not p.scaled:
        # ---- maxima of the scores (the conversion is exact and monotone) -----------------------------
        if last:
            hide(PAST_END)
        sources = (early0, early1) if with_maxima else (None, None)
        for rb in (2, 3) if with_maxima else range(RB):
            for step in maxima(rb, (mx0, mx1), sources):
                step()
            sources = (mx0, mx1)
        score_scales()
        if last:  # the maximum of a scale group starts from -50000
            e.valu(f"v_max_f32_e32 v{mx0}, {ROW_FLOOR}, v{mx0}", [mx0])
            e.valu(f"v_max_f32_e32 v{mx1}, {ROW_FLOOR}, v{mx1}", [mx1])
        e.valu(f"v_mov_b32_e32 v{negm}, {MINUS_U8_OFFSET}", [negm])
        e.valu(f"v_fma_f32 v{mx0}, v{mx0}, v{SC0}, v{negm}", [mx0])
        e.valu(f"v_fma_f32 v{mx1}, v{mx1}, v{SC1}, v{negm}", [mx1])
        e.valu(f"v_max_f32_e32 v{mx0}, v{mx0}, v{mx1}", [mx0])
    else:
        # ---- scaled scores and their maximum -------------------------------------------------------
        score_scales()
        for rb in range(RB):
            for i in range(16):
                register = S[rb] + i
                e.valu(f"v_mul_f32_e32 v{register}, v{register}, v{scale_of(i)}", [register])
        if p.bias:
            e.wait_lds(F)
            e.valu(f"v_or3_b32 v{F}, v{F}, v{F + 1}, v{F + 2}", [F])
            e.valu(f"v_or_b32_e32 v{F}, v{F}, v{F + 3}", [F])
            e.valu(f"v_lshlrev_b32_e32 v{F}, 1, v{F}", [F])  # (a zero of either sign)
            e.valu(f"v_cmp_ne_u32_e32 vcc, 0, v{F}")
            e.nop(4)
            e.ins(f"s_cbranch_vccz {label}_zerorow")
            e.valu(f"v_cndmask_b32_e64 v{F}, 0, 16, {pair(p.halfmask)}", [F])
            e.nop(1)
            for rb in range(RB):
                for b4 in range(4):
                    e.ins(f"ds_read_b128 v[{X + b4 * 4}:{X + b4 * 4 + 3}], v{F} offset:{BIAS_REGION + rb * 128 + b4 * 32}")
                e.ins("s_waitcnt lgkmcnt(0)")
                for i in range(16):
                    e.valu(f"v_add_f32_e32 v{S[rb] + i}, v{S[rb] + i}, v{X + i}", [S[rb] + i])
            e.raw(f"{label}_zerorow:")
        if last:
            hide(NEG_INF)
        e.valu(f"v_mov_b32_e32 v{mx0}, {ROW_FLOOR}", [mx0])
        e.valu(f"v_max_f32_e32 v{mx1}, v{scores[0]}, v{scores[1]}", [mx1])
        for index, at in enumerate(range(2, len(scores), 2)):
            target = mx1 if index & 1 else mx0
            e.valu(f"v_max3_f32 v{target}, v{target}, v{scores[at]}, v{scores[at + 1]}", [target])
        e.valu(f"v_max_f32_e32 v{mx0}, v{mx0}, v{mx1}", [mx0])
        e.valu(f"v_add_f32_e32 v{mx0}, {MINUS_U8_OFFSET}, v{mx0}", [mx0])
    e.valu(f"v_mov_b32_e32 v{mx1}, v{mx0}", [mx1])
    e.nop(2)
    e.valu(f"v_permlane32_swap_b32_e32 v{mx0}, v{mx1}", [mx0, mx1])  # the other half's maximum
    e.nop(2)
    e.valu(f"v_max_f32_e32 v{mx0}, v{mx0}, v{mx1}", [mx0])  # tile maximum - 7.99 of the row
    # ---- online-softmax state: the reference only moves when a tile maximum exceeds it by more than 8
    e.valu(f"v_add_f32_e32 v{tmp}, 0x41000000, v{MRUN}", [tmp])
    e.valu(f"v_cmp_gt_f32_e32 vcc, v{mx0}, v{tmp}")
    e.nop(4)
    e.ins(f"s_cbranch_vccz {label}_keep")
    e.valu(f"v_sub_f32_e32 v{tmp}, v{MRUN}, v{mx0}", [tmp])
    e.valu(f"v_exp_f32_e32 v{tmp}, v{tmp}", [tmp], trans=True)
    e.nop(1)
    e.valu(f"v_cndmask_b32_e32 v{tmp}, 1.0, v{tmp}, vcc", [tmp])
    e.valu(f"v_cndmask_b32_e32 v{MRUN}, v{MRUN}, v{mx0}, vcc", [MRUN])
    e.valu(f"v_mul_f32_e32 v{DPART}, v{DPART}, v{tmp}", [DPART])
    for cb in range(CB):
        for i in range(16):
            e.valu(f"v_mul_f32_e32 v{O[cb] + i}, v{O[cb] + i}, v{tmp}", [O[cb] + i])
    e.raw(f"{label}_keep:")
    e.valu(f"v_sub_f32_e32 v{TSCALE}, v{mx0}, v{MRUN}", [TSCALE])
    e.valu(f"v_exp_f32_e32 v{TSCALE}, v{TSCALE}", [TSCALE], trans=True)

    # ---- exponent arguments in place of the scores -----------------------------------------------------
    if p.scaled:
        for register in scores:
            e.valu(f"v_sub_f32_e32 v{register}, v{register}, v{mx0}", [register])
    else:
        e.valu(f"v_sub_f32_e32 v{negm}, 0, v{mx0}", [negm])
        for rb in range(RB):
            for i in range(16):
                register = S[rb] + i
                e.valu(f"v_fma_f32 v{register}, v{register}, v{scale_of(i)}, v{negm}", [register])
    e.ins("s_waitcnt vmcnt(0)")
    e.ins("s_barrier")  # B
    rowsum, half16 = F, F + 1
    e.valu(f"v_mov_b32_e32 v{rowsum}, 0", [rowsum])
    e.valu(f"v_cndmask_b32_e64 v{half16}, 0, 16, {pair(p.halfmask)}", [half16])

    # ---- scalar side of the next tile: landed by the value product ------------------------------------
    if not last:
        if p.listed:
            address(e, p, p.at, p.ksptr, p.tnext, 4)
            e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.at)}, 0x0")
            e.ins(f"s_add_u32 s{p.index}, s{p.index}, 1")
            e.ins(f"s_min_u32 s{p.index}, s{p.index}, s{p.last}")
            e.ins(f"s_lshl_b32 s{p.at}, s{p.index}, 2")
            e.ins(f"s_add_u32 s{p.at}, s{p.list}, s{p.at}")
            e.ins(f"s_addc_u32 s{p.at + 1}, s{p.list + 1}, 0")
            e.ins(f"s_load_dword s{p.tafter}, {pair(p.at)}, 0x0")
        else:
            add64(e, p.ksptr, 16)
            e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.ksptr)}, 0x0")

    # ---- probabilities, and O^T += scale * (seeds + V^T P^T) in eight channel blocks --------------------
    # Products of the first two channel blocks go between the exponentials as soon as their key block
    # is packed, those of the others between the output updates of the block before: a product behind
    # another one waits for it and holds up everything after it.
    fragments = [(cb, rb) for cb in range(CB) for rb in range(RB)]
    v_slot, next_v = {}, 0
    v_address = [VA, SC0, SC1, F + 3]
    for step in (1, 2, 3):
        e.valu(f"v_xor_b32_e32 v{v_address[step]}, {step * 32}, v{VA}", [v_address[step]])

    def read_value_fragment(cb, rb, at):
        v_slot[cb, rb] = at
        e.ds_read(at, v_address[rb], cb * 32 * KEYS)

    def read_seeds(cb):
        for b4 in range(4):
            e.ds_read(ACC[cb % 3] + b4 * 4, half16, SEED_REGION + cb * 128 + b4 * 32)

    def product(cb, rb):
        block = ACC[cb % 3]
        if rb == 0:
            e.wait_value(block + 12)
        e.wait_value(v_slot[cb, rb])
        e.mfma(block, v_slot[cb, rb], PK + rb * 4, block)

    def pack_group(rb, b4):
        """Four scores -> one register of signed probability bytes, and their sum."""
        registers = [S[rb] + b4 * 4 + r for r in range(4)]
        target = PK + rb * 4 + b4
        for r in range(4):
            e.valu(f"v_exp_f32_e32 v{registers[r]}, v{registers[r]}", [registers[r]], trans=True)
        for r in range(4):
            e.need_trans(registers[r])
            previous = "0" if r == 0 else f"v{target}"
            e.valu(f"v_cvt_pk_u8_f32 v{target}, v{registers[r]}, {r}, {previous}", [target])
        e.valu(f"v_sad_u8 v{rowsum}, v{target}, 0, v{rowsum}", [rowsum])
        e.valu(f"v_xor_b32_e32 v{target}, 0x80808080, v{target}", [target])

    e.ins(f"s_setprio {prio[2]}")
    copies = [] if last else k_copies(e, p, label + "k", F + 2)
    read_seeds(0)
    for rb in range(RB):
        for b4 in range(4):
            if rb == 1 and b4 == 0:    # (the upper half of PK: free until the third block)
                read_value_fragment(0, 0, PK + 8)
            if rb == 1 and b4 == 3:
                product(0, 0)
            if rb == 2 and b4 == 0:
                read_value_fragment(0, 1, VF[1])
                read_value_fragment(0, 2, VF[2])
            if rb == 2 and b4 == 2:
                product(0, 1)
            if rb == 3 and b4 == 0:
                read_seeds(1)
                read_value_fragment(1, 0, VF[0])
                read_value_fragment(1, 1, VF[1])
                read_value_fragment(0, 3, VF[3])
                product(0, 2)
                read_value_fragment(1, 2, VF[2])
            if rb == 3 and b4 > 0:
                product(1, b4 - 1)
            pack_group(rb, b4)
            if copies:
                copies.pop(0)()
    total = F + 2
    read_seeds(2)
    read_value_fragment(2, 0, VF[0])
    read_value_fragment(2, 1, VF[1])
    read_value_fragment(2, 2, VF[2])
    product(0, 3)
    read_value_fragment(1, 3, VF[3])
    e.valu(f"v_cvt_f32_u32_e32 v{total}, v{rowsum}", [total])
    e.valu(f"v_fmac_f32_e32 v{DPART}, v{total}, v{TSCALE}", [DPART])
    if not last and not p.listed:
        add64(e, p.kptr, TILE_BYTES)
        if p.bias:
            add64(e, p.maskptr, KEYS * 4)
    e.ins(f"s_setprio {prio[3]}")

    def update(cb, quarter):
        block = ACC[cb % 3]
        e.need_mfma_result(block)
        for i in range(4 * quarter, 4 * quarter + 4):
            e.valu(f"v_sub_f32_e32 v{block + i}, v{block + i}, v{SEEDVAL}", [block + i])
        for i in range(4 * quarter, 4 * quarter + 4):
            e.valu(f"v_fmac_f32_e32 v{O[cb] + i}, v{block + i}, v{TSCALE}", [O[cb] + i])

    for cb in range(1, CB + 1):
        for rb in range(RB):
            if cb < CB and not (cb == 1 and rb < 3):
                product(cb, rb)
                if cb + 1 < CB and (cb + 1, rb) not in v_slot:
                    read_value_fragment(cb + 1, rb, VF[rb])
            update(cb - 1, rb)
        if cb + 2 < CB:
            read_seeds(cb + 2)


class Counted(Emitter):
    """With a scalar load in flight only a wait for zero proves that an LDS read has landed (the two
    share the counter and scalar loads return in any order)."""

    def __init__(self):
        super().__init__()
        self.scalar_pending = False

    def ins(self, text):
        super().ins(text)
        if text.startswith("s_load"):
            self.scalar_pending = True
        if "lgkmcnt(0)" in text:
            self.scalar_pending = False

    def wait_value(self, dst):
        if dst in self.lds_queue and self.scalar_pending:
            super().ins("s_waitcnt lgkmcnt(0)")
            self.lds_queue, self.scalar_pending = [], False
        else:
            self.wait_lds(dst)


def generate(p, prio):
    e = Counted()
    e.comment("set-up: operands into fixed scalar registers")
    for target, name in ((p.kptr, "kptr"), (p.vptr, "vptr"), (p.sumptr, "sumptr"), (p.ksptr, "ksptr")):
        e.ins(f"s_mov_b64 {pair(target)}, %[{name}]")
    for target, name in ((p.count, "count"), (p.qs2, "qs2"), (p.wave, "wave"), (p.rem, "rem"), (p.remq, "remq")):
        e.ins(f"s_mov_b32 s{target}, %[{name}]")
    e.ins(f"s_lshl_b32 s{p.vstep}, %[padded], 3")
    if p.listed:
        e.ins(f"s_mov_b64 {pair(p.list)}, %[list]")
    if p.bias:
        e.ins(f"s_mov_b64 {pair(p.maskptr)}, %[mask]")
    e.ins(f"s_mov_b32 s{p.halfmask}, 0")
    e.ins(f"s_mov_b32 s{p.halfmask + 1}, -1")
    # this wavefront's copy slots and its share of the sources: eight rows of V, 1 KiB of K a copy
    e.ins(f"s_lshl_b32 s{p.klds}, s{p.wave}, 13")
    e.ins(f"s_add_u32 s{p.kptr}, s{p.kptr}, s{p.klds}")
    e.ins(f"s_addc_u32 s{p.kptr + 1}, s{p.kptr + 1}, 0")
    e.ins(f"s_lshl_b32 s{p.at}, s{p.wave}, 3")
    e.ins(f"s_mul_hi_u32 s{p.kat}, s{p.at}, s{p.vstep}")
    e.ins(f"s_mul_i32 s{p.at}, s{p.at}, s{p.vstep}")
    e.ins(f"s_add_u32 s{p.vptr}, s{p.vptr}, s{p.at}")
    e.ins(f"s_addc_u32 s{p.vptr + 1}, s{p.vptr + 1}, s{p.kat}")
    if p.listed:
        # entries of the first two tiles; the walk reads none behind its last
        e.ins(f"s_mov_b32 s{p.last}, s{p.count}")
        e.ins(f"s_min_u32 s{p.index}, s{p.last}, 1")
        e.ins(f"s_load_dword s{p.tnext}, {pair(p.list)}, 0x0")
        e.ins(f"s_lshl_b32 s{p.at}, s{p.index}, 2")
        e.ins(f"s_add_u32 s{p.at}, s{p.list}, s{p.at}")
        e.ins(f"s_addc_u32 s{p.at + 1}, s{p.list + 1}, 0")
        e.ins(f"s_load_dword s{p.tafter}, {pair(p.at)}, 0x0")
        e.ins("s_waitcnt lgkmcnt(0)")
        address(e, p, p.at, p.ksptr, p.tnext, 4)
        e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.at)}, 0x0")
    else:
        e.ins(f"s_load_dwordx4 s[{p.ks}:{p.ks + 3}], {pair(p.ksptr)}, 0x0")
    e.ins(f"v_mov_b32_e32 v{SEEDVAL}, 0x4b400000")
    for piece in k_copies(e, p, "Lrisa_first_%=", X):
        piece()
    if not p.listed:
        add64(e, p.kptr, TILE_BYTES)
        if p.bias:
            add64(e, p.maskptr, KEYS * 4)
    e.ins(f"s_cmp_eq_u32 s{p.count}, 0")
    e.ins("s_cbranch_scc1 Lrisa_last_%=")
    e.raw("Lrisa_loop_%=:")
    tile_body(e, p, False, prio, "Lrisa_a_%=")
    e.ins(f"s_sub_u32 s{p.count}, s{p.count}, 1")
    e.ins(f"s_cmp_lg_u32 s{p.count}, 0")
    e.ins("s_cbranch_scc1 Lrisa_loop_%=")
    e.raw("Lrisa_last_%=:")
    tile_body(e, p, True, prio, "Lrisa_b_%=")
    e.ins("s_setprio 0")
    return e


PROGRAMS = (
    Program("raw", scaled=False),
    Program("scaled", scaled=True),
    Program("bias", scaled=True, bias=True),
    Program("bias_listed", scaled=True, bias=True, listed=True),
)


def operands(p):
    """(outputs, inputs) as (constraint, C++ expression) pairs, and the named scalar inputs."""
    block = lambda first, count: f"{{v[{first}:{first + count - 1}]}}" if count > 1 else f"{{v{first}}}"
    outputs = [(block(O[cb], 16), f"out[{cb}]") for cb in range(CB)]
    outputs += [(block(MRUN, 1), "m_run"), (block(DPART, 1), "d_part")]
    inputs = [(block(Q[kk], 4), f"qreg[{kk}]") for kk in range(KK)]
    inputs += [(block(QSCALE, 1), "q_scale"), (block(KA, 1), "k_address"), (block(VA, 1), "v_address"),
               (block(VC, 1), "v_share"), (block(KC, 1), "k_share")]
    named = [("kptr", "k_base"), ("vptr", "v_base"), ("sumptr", "sum_base"), ("ksptr", "ks_base"),
             ("count", "count"), ("wave", "wave"), ("qs2", "p.sm2"), ("padded", "p.padded"),
             ("rem", "keys_left"), ("remq", "keys_to_query")]
    if p.listed:
        named.append(("list", "indices"))
    if p.bias:
        named.append(("mask", "bias_base"))
    return outputs, inputs, named


def render(p, prio=PRIORITIES):
    """The asm statement as the include file holds it."""
    e = generate(p, prio)
    outputs, inputs, named = operands(p)
    text = "asm volatile(\n" + "".join('"{}\\n\\t"\n'.format(line) for line in e.lines)
    text += "    : " + ", ".join(f'"+{c}"({x})' for c, x in outputs + [i for i in inputs if i[1] in ("v_share", "k_share")]) + "\n"
    inputs = [i for i in inputs if i[1] not in ("v_share", "k_share")]
    text += "    : " + ", ".join(f'"{c}"({x})' for c, x in inputs) + ",\n"
    text += "      " + ", ".join(f'[{n}] "s"({x})' for n, x in named) + "\n"
    pinned = set(range(0, 128)) | set(range(Q[0], Q[0] + 32)) | {MRUN, DPART, QSCALE, KA, VA, VC, KC}
    clobbered = [f"v{r}" for r in range(LAST_VGPR + 1) if r not in pinned]
    clobbered += [f"s{r}" for r in range(FIRST_SGPR, p.next_sgpr)] + ["vcc", "scc", "m0", "memory"]
    text += "    : " + ", ".join(f'"{name}"' for name in clobbered) + ");\n"
    return text


def main():
    parser = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    parser.add_argument("--outdir", type=pathlib.Path, default=pathlib.Path(__file__).resolve().parent)
    args = parser.parse_args()
    for program in PROGRAMS:
        (args.outdir / f"d256_loop_{program.name}.inc").write_text(render(program))


if __name__ == "__main__":
    main()
