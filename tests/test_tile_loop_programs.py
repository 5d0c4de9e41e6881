"""The tile loops of gen_tile_loops.py checked on the CPU, as tests/test_dense_loop_program.py checks
the raw-score ones: the committed text is what the generator writes, and an interpreter of the
addresses (scalar side, M0, EXEC, address registers) and wait counters compares every copy, LDS
read, matrix-instruction operand and scalar load with what the C++ tile loop does.  It asserts that
no instruction touches a register an LDS read or scalar load is still to fill, that copies stay
inside the tiles they name, and the wait states behind matrix instructions."""

import importlib.util
import random
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "risaattention_amd" / "csrc"
K0, V0, SUM0, KS0, LIST0, MASK0 = 0x10000000, 0x20000000, 0x30000000, 0x40000000, 0x50000000, 0x60000000
LANES = range(64)
FULL = (1 << 64) - 1


def generator():
    spec = importlib.util.spec_from_file_location("gen_tile_loops", CSRC / "gen_tile_loops.py")
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


GEN = generator()


def swizzled(row, chunk, rowbytes):
    chunks = rowbytes // 16
    return row * rowbytes + ((chunk ^ ((row // (256 // rowbytes)) & (chunks - 1))) << 4)


def source_offset(wave, copies, i, lane, rowbytes, pitch):
    """k_source_offset / v_source_offset of attention_kernel.hpp."""
    chunks = rowbytes // 16
    slot = (wave * copies + i) * 64 + lane
    row, phys = slot // chunks, slot % chunks
    return row * pitch + (phys ^ ((row // (256 // rowbytes)) & (chunks - 1))) * 16


def mask_offset(wave, i, lane, row_bytes):
    """issue_mask_tile of attention_kernel.hpp, 4-byte elements, 64-key tiles."""
    index = (wave * 8 + i) * 64 + lane
    row = index // 16
    return row * row_bytes + ((index % 16) ^ (row & 15)) * 16


def interpret(program, text, vreg, named, memory):
    lines = [re.match(r'"(.*)\\n\\t"', line).group(1).split(";")[0].strip() for line in text.splitlines() if line.startswith('"')]
    lines = [line for line in lines if line]
    labels = {line[:-1]: index for index, line in enumerate(lines) if line.endswith(":")}
    sreg, state = {"vcc": 0}, {"exec": FULL, "scc": 0}
    pending_lds, pending_scalar = [], []
    fragment, written, clock = {}, {}, 0
    events, phase, pc = [], 0, 0

    def registers(token):
        single = re.fullmatch(r"([sv])(\d+)", token)
        if single:
            return single.group(1), [int(single.group(2))]
        block = re.fullmatch(r"([sv])\[(\d+):(\d+)\]", token)
        return (block.group(1), list(range(int(block.group(2)), int(block.group(3)) + 1))) if block else (None, [])

    def value(token):
        if token.startswith("%["):
            return named[token[2:-1]]
        if token == "exec":
            return state["exec"]
        if token == "m0":
            return sreg["m0"]
        kind, numbers = registers(token)
        if kind == "s":
            return sum(sreg.get(n, 0) << (32 * at) for at, n in enumerate(numbers))
        return int(token, 0) & FULL

    def assign(token, result):
        if token == "exec":
            state["exec"] = result & FULL
        elif token == "m0":
            sreg["m0"] = result & 0xFFFFFFFF
        else:
            for at, n in enumerate(registers(token)[1]):
                sreg[n] = result >> (32 * at) & 0xFFFFFFFF

    def lane_values(token):
        kind, numbers = registers(token)
        return vreg[numbers[0]] if kind == "v" else [value(token) & 0xFFFFFFFF] * 64

    steps = 0
    while pc < len(lines):
        steps += 1
        assert steps < 3_000_000, "the loop does not end"
        line = lines[pc]
        pc += 1
        if line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        if op == "s_nop":
            clock += int(rest) + 1
            continue
        clock += 1
        args = [a.strip() for a in re.split(r",(?![^\[]*\])", rest)] if rest else []
        touched = {(kind, n) for token in re.findall(r"[sv]\[\d+:\d+\]|\b[sv]\d+\b", rest) for kind, ns in [registers(token)] for n in ns}
        busy = {("v", n) for block in pending_lds for n in block} | {("s", n) for block in pending_scalar for n in block}
        if op != "s_waitcnt":
            assert not touched & busy, f"still to be filled: {line}"
        low = lambda at: value(args[at]) & 0xFFFFFFFF
        if op == "s_barrier":
            assert not pending_lds and not pending_scalar
            phase += 1
            written.clear()
        elif op == "s_waitcnt":
            count = re.search(r"lgkmcnt\((\d+)\)", rest)
            if count and int(count.group(1)) == 0:
                pending_lds, pending_scalar = [], []
            elif count:
                assert not pending_scalar, f"a partial wait with a scalar load in flight: {line}"
                pending_lds = pending_lds[max(0, len(pending_lds) - int(count.group(1))):]
        elif op in ("s_mov_b32", "s_mov_b64", "s_movk_i32"):
            assign(args[0], value(args[1]))
        elif op == "v_readfirstlane_b32":
            assign(args[0], lane_values(args[1])[0])
        elif op == "s_lshl_b32":
            assign(args[0], low(1) << low(2))
        elif op in ("s_add_u32", "s_addc_u32"):
            total = low(1) + low(2) + (state["scc"] if op == "s_addc_u32" else 0)
            state["scc"] = total >> 32
            assign(args[0], total)
        elif op == "s_sub_u32":
            state["scc"] = int(low(1) < low(2))
            assign(args[0], low(1) - low(2))
        elif op == "s_min_u32":
            assign(args[0], min(low(1), low(2)))
        elif op == "s_mul_i32":
            assign(args[0], low(1) * low(2))
        elif op == "s_mul_hi_u32":
            assign(args[0], low(1) * low(2) >> 32)
        elif op in ("s_cmp_eq_u32", "s_cmp_lg_u32"):
            state["scc"] = int((low(0) == low(1)) == (op == "s_cmp_eq_u32"))
        elif op == "s_cbranch_scc1":
            pc = labels[args[0]] if state["scc"] else pc
        elif op == "s_cbranch_vccz":
            # both sides in turn: the rescale block touches no memory, the bias block reads its row
            state["taken"] = not state.get("taken", False)
            pc = labels[args[0]] if state["taken"] else pc
        elif op.startswith("s_load_dword"):
            address = value(args[1]) + int(args[2], 0)
            numbers = registers(args[0])[1]
            events.append((phase, "sload", (address, len(numbers))))
            for at, n in enumerate(numbers):
                sreg[n] = memory.get(address + 4 * at, 0)
            pending_scalar.append(numbers)
        elif op == "global_load_lds_dwordx4":
            assert "offset" not in rest
            base, offsets = value(args[1]), lane_values(args[0])
            events.append((phase, "copy", [(sreg["m0"] + 16 * l, base + offsets[l]) for l in LANES if state["exec"] >> l & 1]))
        elif op == "ds_read_b128":
            address, offset = re.fullmatch(r"(v\d+) offset:(\d+)", args[1]).groups()
            assert int(offset) < 65536
            block = registers(args[0])[1]
            addresses = tuple(a + int(offset) for a in lane_values(address))
            events.append((phase, "read", (block[0], addresses)))
            pending_lds.append(block)
            for n in block:
                vreg.pop(n, None)
                assert clock - written.get(n, -100) >= 12
            fragment[block[0]] = addresses
        elif op == "v_mfma_i32_32x32x32_i8":
            blocks = [registers(arg)[1][0] for arg in args]
            events.append((phase, "mfma", (blocks[0], fragment[blocks[1]], blocks[2], blocks[3])))
            for n in registers(args[0])[1]:
                written[n] = clock
        elif op.startswith("v_"):
            for kind, n in touched:
                if kind == "v":
                    assert clock - written.get(n, -100) >= 12, f"matrix result too early: {line}"
            kind, numbers = registers(args[0])
            known = None
            sources = args[1:]
            if op.startswith(("v_xor_b32", "v_xad_u32", "v_mbcnt_lo", "v_lshlrev_b32", "v_and_b32", "v_lshl_add_u32")):
                readable = all(registers(t)[0] != "v" or registers(t)[1][0] in vreg for t in sources)
                if readable:
                    a = [lane_values(t) for t in sources]
                    known = {
                        "v_xor_b32_e32": lambda l: a[0][l] ^ a[1][l],
                        "v_and_b32_e32": lambda l: a[0][l] & a[1][l],
                        "v_xad_u32": lambda l: (a[0][l] ^ a[1][l]) + a[2][l] & 0xFFFFFFFF,
                        "v_mbcnt_lo_u32_b32": lambda l: min(l, 32),
                        "v_lshlrev_b32_e32": lambda l: a[1][l] << a[0][l] & 0xFFFFFFFF,
                        "v_lshl_add_u32": lambda l: (a[0][l] << a[1][l]) + a[2][l] & 0xFFFFFFFF,
                    }[op]
                    known = [known(l) for l in LANES]
            if kind == "v":
                for n in numbers:
                    vreg.pop(n, None)
                    fragment.pop(n, None)
                if known:
                    vreg[numbers[0]] = known
            if op.startswith("v_permlane32_swap"):
                vreg.pop(registers(args[1])[1][0], None)
        elif op != "s_setprio":
            raise AssertionError(f"instruction the interpreter does not know: {line}")
    return events, phase


@pytest.mark.parametrize("program", GEN.PROGRAMS, ids=lambda p: p.name)
def test_generated_text_is_committed(program):
    text = GEN.render(program)
    assert (CSRC / f"tile_loop_{program.name}.inc").read_text() == text
    assert '"v255"' not in text and "s_store" not in text and "s_dcache" not in text and "s_atomic" not in text
    assert {p.stem for p in CSRC.glob("tile_loop_*.inc")} == {f"tile_loop_{p.name}" for p in GEN.PROGRAMS}


@pytest.mark.parametrize("walk", [1, 2, 5, 16])
@pytest.mark.parametrize("program", GEN.PROGRAMS, ids=lambda p: p.name)
def test_memory_accesses_match_the_compiled_loop(program, walk):
    p = program
    dim, keys, copies, stage_bytes = p.dim, p.keys, p.dim * p.keys // 4096, 2 * p.dim * p.keys + 4 * (p.dim + p.keys)
    tiles = walk + 3
    padded, row_bytes = tiles * keys, (tiles * keys + 20) * 4
    listed = sorted(random.Random(walk).sample(range(tiles), walk + 1)) if p.listed else list(range(walk + 1))
    memory = {LIST0 + 4 * i: tile for i, tile in enumerate(listed)}
    half, l32 = [l // 32 for l in LANES], [l % 32 for l in LANES]
    text = GEN.render(p)
    for wave in range(4):
        vreg = {}
        k_address = [[swizzled(l32[l], kk * 2 + half[l], dim) for l in LANES] for kk in range(p.kk)]
        v_address = [[swizzled(l32[l], rb * 2 + half[l], keys) for l in LANES] for rb in range(p.rb)]
        if p.ka is not None:
            vreg[p.ka] = k_address[0]
        else:
            vreg.update(zip(p.KA, k_address))
        vreg.update(zip(p.VA, v_address))
        vreg[p.seedaddr] = [h * 16 + 2048 for h in half]
        for i, register in enumerate(p.KC):
            vreg[register] = [source_offset(wave, copies, i, l, dim, dim) - (wave * copies + i) * 1024 for l in LANES]
        rows = 1024 // keys
        for i, register in enumerate(p.VC):
            vreg[register] = [source_offset(wave, copies, i, l, keys, padded) - (wave * copies + i) * rows * padded for l in LANES]
        if p.mask == "f32":
            vreg[p.maddr] = [2 * stage_bytes + (wave * 32 + l32[l]) * 256 + ((half[l] ^ l32[l] & 15) << 4) for l in LANES]
            vreg[p.mch] = [(l % 16 ^ l // 16) << 4 for l in LANES]
            vreg[p.mrow] = [l // 16 * row_bytes for l in LANES]
        ahead = 0 if p.listed else 1
        mask = {None: 0, "f32": MASK0 + keys * 4 + wave * 32 * row_bytes, "bias": MASK0 + ahead * keys * 4, "lanes": MASK0}[p.mask]
        named = {"kptr": K0 + ahead * keys * dim, "vptr": V0 + ahead * keys, "sumptr": SUM0 + ahead * dim * 4, "ksptr": KS0,
                 "count": walk, "wave": wave, "qs2": 0x3F800000, "padded": padded, "list": LIST0, "mask": mask,
                 "maskstep": 4 * row_bytes}
        events, phases = interpret(p, text, vreg, named, memory)
        assert phases == walk

        def of(phase, kind):
            return [event[2] for event in events if event[0] == phase and event[1] == kind]

        words = lambda tile, block: [(MASK0 + tile * 256 + block * 128 + at, 16) for at in (0, 64)]
        first = [(LIST0, 2)] if p.listed else []
        assert of(0, "sload") == first + [(KS0 + 16 * listed[0], 4)] + (words(listed[0], 0) if p.mask == "lanes" else [])
        assert not of(0, "copy") and not of(0, "read") and not of(0, "mfma")
        for index in range(walk):
            stage, other, following = index & 1, index & 1 ^ 1, listed[index + 1]
            copied = []
            for i in range(copies):
                for l in LANES:
                    slot = other * stage_bytes + (wave * copies + i) * 1024 + 16 * l
                    copied.append((slot, K0 + following * keys * dim + source_offset(wave, copies, i, l, dim, dim)))
                    copied.append((slot + dim * keys, V0 + following * keys + source_offset(wave, copies, i, l, keys, padded)))
            region = other * stage_bytes + 2 * dim * keys
            if wave == 0:
                copied += [(region + 16 * l, SUM0 + following * dim * 4 + 16 * l) for l in range(dim // 4)]
            if wave == 1 and p.mask == "bias":
                copied += [(region + dim * 4 + 16 * l, MASK0 + following * keys * 4 + 16 * l) for l in range(keys // 4)]
            if p.mask == "f32" and index + 1 < walk:
                copied += [(2 * stage_bytes + (wave * 8 + i) * 1024 + 16 * l,
                            MASK0 + following * keys * 4 + mask_offset(wave, i, l, row_bytes)) for i in range(8) for l in LANES]
            assert sorted(c for copy in of(index + 1, "copy") for c in copy) == sorted(copied), (wave, index)
            base, seeds = stage * stage_bytes, stage * stage_bytes + 2 * dim * keys
            k_fragment = lambda rb, kk: tuple(base + swizzled(rb * 32 + l32[l], kk * 2 + half[l], dim) for l in LANES)
            v_fragment = lambda cb, rb: tuple(base + dim * keys + swizzled(cb * 32 + l32[l], rb * 2 + half[l], keys) for l in LANES)
            reads = [(p.ACC[kk] + rb * 4, k_fragment(rb, kk)) for kk in range(p.kk) for rb in range(p.rb)]
            reads += [(p.ACC[cb] + b4 * 4, tuple(seeds + (cb * 32 + b4 * 8 + h * 4) * 4 for h in half)) for cb in range(p.cb) for b4 in range(4)]
            reads += [(p.VF[cb], v_fragment(cb, rb)) for cb in range(p.cb) for rb in range(p.rb)]
            quads = [(rb, b4) for rb in range(p.rb) for b4 in range(4)]
            if p.mask == "f32":
                for rb, b4 in quads:
                    chunk = [rb * 8 + b4 * 2 + h for h in half]
                    reads.append((p.M + rb * 16 + b4 * 4, tuple(2 * stage_bytes + (wave * 32 + l32[l]) * 256 + ((chunk[l] ^ l32[l] & 15) << 4) for l in LANES)))
            issued = of(index + 1, "read")
            if p.mask == "bias":
                row = seeds + dim * 4
                reads.append((p.PK[0], tuple(row + (min(l, 32) & keys // 4 - 1) * 16 for l in LANES)))
                terms = [addresses for _, addresses in issued if min(addresses) >= row and addresses != reads[-1][1]]
                assert terms in ([], [tuple(row + (rb * 32 + b4 * 8 + h * 4) * 4 for h in half) for rb, b4 in quads])
                issued = [read for read in issued if read[1] not in terms]
            assert sorted(issued) == sorted(reads), (wave, index)
            products = of(index + 1, "mfma")
            assert len(products) == 2 * p.rb * p.kk
            for rb in range(p.rb):
                assert [m for m in products if m[0] == p.S[rb]] == [
                    (p.S[rb], k_fragment(rb, kk), p.Q[kk], p.S[rb] if kk else p.SEEDS) for kk in range(p.kk)]
            for cb in range(p.cb):
                assert [m for m in products if m[0] == p.ACC[cb]] == [
                    (p.ACC[cb], v_fragment(cb, rb), p.PK[rb & 1], p.ACC[cb]) for rb in range(p.rb)]
            loads = [(KS0 + 16 * following, 4)]
            if p.listed:
                own = words(listed[index], 1) if p.mask == "lanes" else []
                ahead_words = words(following, 0) if p.mask == "lanes" else []
                loads = own + loads + ahead_words + [(LIST0 + 4 * min(index + 2, walk), 1)]
            assert of(index + 1, "sload") == loads, (wave, index)
