"""Runs a hand-scheduled program (the text of a generated asm statement) on the CPU: the wavefronts of
one workgroup with their registers, LDS and the global memory they may touch, values included.

What it refuses: an access outside the given memory, an LDS read of bytes a copy is still to fill or
that nothing has filled, a register touched while an LDS read or scalar load is to fill it, a barrier
reached with loads in flight or not by every wavefront, vector instructions on a matrix result before it
is there, and vector instructions that read a comparison's scalar result less than two wait states behind
it (what the compiler leaves between its own: nothing in hardware holds the reader back)."""

import re

import numpy as np

LANES = np.arange(64)
MATRIX_RESULT_STATES = 12  # wait states between an 8-pass matrix instruction and a vector one on its result
COMPARISON_STATES = 2  # wait states between a vector comparison and a vector instruction that reads its result


class Memory:
    """Global memory: byte arrays at addresses, every access checked."""

    def __init__(self):
        self.segments = []
        self.next = 0x10000000

    def add(self, array):
        data = np.ascontiguousarray(array).view(np.uint8).reshape(-1)
        base, self.next = self.next, self.next + (data.size + 0xFFFFF & ~0xFFFFF) + 0x100000
        self.segments.append((base, data))
        return base

    def read(self, address, count):
        for base, data in self.segments:
            if base <= address and address + count <= base + data.size:
                return data[address - base:address - base + count]
        raise AssertionError(f"read of {count} bytes at {address:#x}")


class Wave:
    def __init__(self, program, memory, lds, vector, named):
        self.lines = [re.match(r'"(.*)\\n\\t"', line).group(1).split(";")[0].strip() for line in program.splitlines() if line.startswith('"')]
        self.lines = [line for line in self.lines if line]
        self.labels = {line[:-1]: at for at, line in enumerate(self.lines) if line.endswith(":")}
        self.memory, self.lds, self.named = memory, lds, named
        self.v = np.zeros((256, 64), np.uint32)
        for register, values in vector.items():
            self.v[register] = np.broadcast_to(np.asarray(values).astype(np.uint32), 64)
        self.s, self.vcc, self.scc, self.exec, self.m0 = {}, np.zeros(64, bool), 0, np.ones(64, bool), 0
        self.pending_lds, self.pending_scalar, self.pending_copies, self.written, self.clock = [], [], [], {}, 0
        self.compared = {}  # scalar registers ("vcc" by name) -> when a vector comparison wrote them

    # ---- operands ------------------------------------------------------------------------------------
    @staticmethod
    def registers(token):
        single = re.fullmatch(r"([sv])(\d+)", token)
        if single:
            return single.group(1), [int(single.group(2))]
        block = re.fullmatch(r"([sv])\[(\d+):(\d+)\]", token)
        return (block.group(1), list(range(int(block.group(2)), int(block.group(3)) + 1))) if block else (None, [])

    def scalar(self, token):
        if token.startswith("%["):
            return self.named[token[2:-1]]
        if token == "m0":
            return self.m0
        kind, numbers = self.registers(token)
        if kind == "s":
            return sum(self.s[n] << (32 * at) for at, n in enumerate(numbers))
        if re.fullmatch(r"-?\d+\.\d+", token):
            return int(np.float32(token).view(np.uint32))
        return int(token, 0) & 0xFFFFFFFFFFFFFFFF

    def assign(self, token, result):
        if token == "m0":
            self.m0 = result & 0xFFFFFFFF
        elif token == "exec":
            self.exec = np.array([result >> l & 1 for l in range(64)], bool)
        else:
            for at, n in enumerate(self.registers(token)[1]):
                self.s[n] = result >> (32 * at) & 0xFFFFFFFF

    def vector(self, token):
        kind, numbers = self.registers(token)
        return self.v[numbers[0]] if kind == "v" else np.full(64, self.scalar(token) & 0xFFFFFFFF, np.uint32)

    def lanes_of(self, token):
        mask = None if token == "vcc" else self.scalar(token)
        return self.vcc if mask is None else np.array([mask >> l & 1 for l in range(64)], bool)

    # ---- execution: yields at every barrier -------------------------------------------------------------
    def run(self):
        pc = steps = 0
        f = lambda x: x.view(np.float32)
        u = lambda x: np.asarray(x, np.float32).view(np.uint32)
        i = lambda x: x.view(np.int32)
        with np.errstate(all="ignore"):
            while pc < len(self.lines):
                steps += 1
                assert steps < 400_000, "the program does not end"
                line = self.lines[pc]
                pc += 1
                if line.endswith(":"):
                    continue
                op, _, rest = line.partition(" ")
                if op == "s_nop":
                    self.clock += int(rest) + 1
                    continue
                self.clock += 1
                rest, _, offset = rest.partition(" offset:")
                args = [a.strip() for a in re.split(r",(?![^\[]*\])", rest)] if rest else []
                touched = {(k, n) for a in args for k, ns in [self.registers(a)] for n in ns}
                busy = {("v", n) for block, _ in self.pending_lds for n in block} | {("s", n) for block in self.pending_scalar for n in block}
                assert op == "s_waitcnt" or not touched & busy, f"still to be filled: {line}"
                if op == "s_barrier":
                    assert not (self.pending_lds or self.pending_scalar or self.pending_copies), "loads in flight at a barrier"
                    yield
                elif op == "s_waitcnt":
                    if "vmcnt(0)" in rest:
                        for places, data in self.pending_copies:
                            self.lds.data[places], self.lds.valid[places] = data, True
                        self.pending_copies = []
                    count = re.search(r"lgkmcnt\((\d+)\)", rest)
                    if count:
                        left = int(count.group(1))
                        assert left == 0 or not self.pending_scalar, line
                        landed = self.pending_lds[:len(self.pending_lds) - left] if left else self.pending_lds
                        for block, data in landed:
                            self.v[block] = data
                        self.pending_lds = self.pending_lds[len(landed):]
                        if left == 0:
                            self.pending_scalar = []
                elif op in ("s_mov_b32", "s_mov_b64", "s_movk_i32"):
                    self.assign(args[0], FULL if args[0] == "exec" and args[1] == "-1" else self.scalar(args[1]))
                elif op == "v_readfirstlane_b32":
                    self.assign(args[0], int(self.vector(args[1])[0]))
                elif op.startswith("s_load_dword"):
                    numbers = self.registers(args[0])[1]
                    data = self.memory.read(self.scalar(args[1]) + int(args[2], 0), 4 * len(numbers)).view(np.uint32)
                    for n, value in zip(numbers, data):
                        self.s[n] = int(value)
                    self.pending_scalar.append(numbers)
                elif op.startswith("s_cbranch"):
                    taken = self.scc if op == "s_cbranch_scc1" else not self.vcc.any() if op == "s_cbranch_vccz" else None
                    pc = self.labels[args[0]] if taken else pc
                elif op.startswith("s_") and op != "s_setprio":
                    a, b = (self.scalar(t) & 0xFFFFFFFF for t in args[-2:])
                    if op.startswith("s_cmp"):
                        self.scc = {"eq": a == b, "lg": a != b, "ge": a >= b}[op[6:8]]
                        continue
                    carry = int(self.scc) if op == "s_addc_u32" else 0
                    result = {"s_add_u32": a + b, "s_addc_u32": a + b + carry, "s_sub_u32": a - b, "s_lshl_b32": a << (b & 31),
                              "s_min_u32": min(a, b), "s_mul_i32": a * b, "s_mul_hi_u32": a * b >> 32}[op]
                    if op in ("s_add_u32", "s_addc_u32"):
                        self.scc = result >> 32
                    elif op == "s_sub_u32":
                        self.scc = a < b
                    self.assign(args[0], result & 0xFFFFFFFF)
                elif op == "global_load_lds_dwordx4":
                    assert not offset
                    base, lanes = self.scalar(args[1]), np.flatnonzero(self.exec)
                    data = np.concatenate([self.memory.read(base + int(self.vector(args[0])[l]), 16) for l in lanes])
                    places = (self.m0 + 16 * lanes[:, None] + np.arange(16)).reshape(-1)
                    assert self.m0 % 4 == 0 and places.max() < self.lds.data.size
                    self.lds.valid[places] = False
                    self.pending_copies.append((places, data))
                elif op == "ds_read_b128":
                    block = self.registers(args[0])[1]
                    assert int(offset) < 65536 and block[0] % 2 == 0
                    places = self.vector(args[1]).astype(np.int64)[:, None] + int(offset) + np.arange(16)
                    assert self.lds.valid[places].all(), f"LDS bytes not there: {line}"
                    for n in block:
                        assert self.clock - self.written.get(n, -100) >= MATRIX_RESULT_STATES, line
                    self.pending_lds.append((block, self.lds.data[places].reshape(64, 4, 4).view(np.uint32)[..., 0].T.copy()))
                elif op == "v_mfma_i32_32x32x32_i8":
                    d, a, b, c = (self.registers(t)[1] for t in args)
                    assert not set(d) & (set(a) | set(b)) and (d == c or not set(d) & set(c)), line
                    rows = lambda block: self.v[block].T.copy().view(np.int8).reshape(2, 32, 16).transpose(1, 0, 2).reshape(32, 32).astype(np.int32)
                    product = rows(a) @ rows(b).T  # [row of A, column]
                    result = np.empty((16, 64), np.int32)
                    for r in range(16):
                        for half in (0, 1):
                            result[r, 32 * half:32 * half + 32] = product[8 * (r // 4) + 4 * half + r % 4]
                    self.v[d] = (result + i(self.v[c])).view(np.uint32)
                    self.written.update({n: self.clock for n in d})
                elif op == "v_permlane32_swap_b32_e32":
                    x, y = self.registers(args[0])[1][0], self.registers(args[1])[1][0]
                    self.v[x, 32:], self.v[y, :32] = self.v[y, :32].copy(), self.v[x, 32:].copy()
                elif op.startswith("v_cmp"):
                    self.check(touched, line)
                    a, b = self.vector(args[1]), self.vector(args[2])
                    result = {"gt_f32": f(a) > f(b), "lt_i32": i(a) < i(b), "ne_u32": a != b}[re.sub(r"v_cmp_|_e\d\d", "", op)]
                    if args[0] == "vcc":
                        self.vcc = result
                    else:
                        self.assign(args[0], int(sum(int(bit) << lane for lane, bit in enumerate(result))))
                    self.compared.update({n: self.clock for n in self.registers(args[0])[1] or ["vcc"]})
                elif op.startswith("v_"):
                    self.check(touched, line)
                    for n in {n for k, n in touched if k == "s"} | {"vcc"} & set(args):
                        assert self.clock - self.compared.get(n, -100) > COMPARISON_STATES, f"comparison's result too early: {line}"
                    x = [self.vector(t) for t in args[1:] if not re.fullmatch(r"s\[\d+:\d+\]|vcc", t)]
                    if op.startswith("v_cndmask"):
                        result = np.where(self.lanes_of(args[3]), x[1], x[0])
                    elif op == "v_cvt_pk_u8_f32":
                        byte, shift = np.clip(np.rint(np.nan_to_num(f(x[0]), nan=0.0, posinf=255.0)), 0, 255).astype(np.uint32), 8 * int(x[1][0])
                        result = x[2] & ~np.uint32(0xFF << shift) | byte << np.uint32(shift)
                    elif op == "v_sad_u8":
                        result = np.abs(x[0].view(np.uint8).astype(np.int32) - x[1].view(np.uint8)).reshape(64, 4).sum(1) + x[2]
                    elif op in ("v_fma_f32", "v_fmac_f32_e32"):
                        addend = x[2] if op == "v_fma_f32" else self.vector(args[0])
                        # (the double product is exact, so only the rare double rounding differs)
                        result = u((f(x[0]).astype(np.float64) * f(x[1]) + f(addend)).astype(np.float32))
                    else:
                        result = {
                            "v_mov_b32_e32": lambda: x[0],
                            "v_add_f32_e32": lambda: u(f(x[0]) + f(x[1])), "v_sub_f32_e32": lambda: u(f(x[0]) - f(x[1])),
                            "v_mul_f32_e32": lambda: u(f(x[0]) * f(x[1])), "v_max_f32_e32": lambda: u(np.fmax(f(x[0]), f(x[1]))),
                            "v_max3_f32": lambda: u(np.fmax(np.fmax(f(x[0]), f(x[1])), f(x[2]))),
                            "v_max_i32_e32": lambda: np.maximum(i(x[0]), i(x[1])), "v_min_i32_e32": lambda: np.minimum(i(x[0]), i(x[1])),
                            "v_max3_i32": lambda: np.maximum(np.maximum(i(x[0]), i(x[1])), i(x[2])),
                            "v_exp_f32_e32": lambda: u(np.exp2(f(x[0]).astype(np.float64))), "v_cvt_f32_u32_e32": lambda: u(x[0]),
                            "v_add_u32_e32": lambda: x[0] + x[1], "v_sub_u32_e32": lambda: x[0] - x[1],
                            "v_xor_b32_e32": lambda: x[0] ^ x[1], "v_and_b32_e32": lambda: x[0] & x[1], "v_or_b32_e32": lambda: x[0] | x[1],
                            "v_or3_b32": lambda: x[0] | x[1] | x[2],
                            "v_lshlrev_b32_e32": lambda: x[1] << (x[0] & 31), "v_lshrrev_b32_e32": lambda: x[1] >> (x[0] & 31),
                            "v_lshl_add_u32": lambda: (x[0] << (x[1] & 31)) + x[2],
                            "v_mbcnt_lo_u32_b32": lambda: np.minimum(LANES, 32) + x[1],
                            "v_mbcnt_hi_u32_b32": lambda: np.maximum(LANES - 32, 0) + x[1],
                        }[op]()
                    target = self.registers(args[0])[1][0]
                    result = np.asarray(result)
                    self.v[target] = result if result.dtype == np.uint32 else result.astype(np.int64).astype(np.uint32)
                else:
                    assert op == "s_setprio", f"instruction the emulator does not know: {line}"

    def check(self, touched, line):
        for kind, n in touched:
            assert kind != "v" or self.clock - self.written.get(n, -100) >= MATRIX_RESULT_STATES, f"matrix result too early: {line}"


FULL = (1 << 64) - 1


class Lds:
    def __init__(self, size):
        self.data, self.valid = np.zeros(size, np.uint8), np.zeros(size, bool)


def run_workgroup(waves, order=None):
    """All wavefronts from barrier to barrier, in the given order within each interval."""
    running = [wave.run() for wave in waves]
    order = list(order or range(len(waves)))
    while running:
        ended = []
        for at in order:
            try:
                next(running[at])
                ended.append(False)
            except StopIteration:
                ended.append(True)
        assert all(ended) or not any(ended), "a barrier some wavefronts do not reach"
        if all(ended):
            return
        order = order[::-1]
