"""The tile walks of head dim 256 (gen_d256_loops.py) on the CPU: the committed text is what the
generator writes, and each program, run by an emulator on the operands of one query block, gives the
oracle's output: tile counts from one, keys past the end, queries past the end, causal limits, scales
of any sign, additive rows and tile lists."""

import importlib.util
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import attention
from risaattention_amd.layout import pack_values
from tests.wave_emulator import Lds, Memory, Wave, run_workgroup

CSRC = Path(__file__).resolve().parents[1] / "risaattention_amd" / "csrc"
DIM, KEYS, SEED_BITS = 256, 128, 0x4B400000
LANE = np.arange(64)
HALF, L32 = LANE // 32, LANE % 32


def generator():
    spec = importlib.util.spec_from_file_location("gen_d256_loops", CSRC / "gen_d256_loops.py")
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


GEN = generator()
PROGRAMS = {p.name: p for p in GEN.PROGRAMS}


@pytest.mark.parametrize("program", GEN.PROGRAMS, ids=lambda p: p.name)
def test_generated_text_is_committed(program):
    text = GEN.render(program)
    assert (CSRC / f"d256_loop_{program.name}.inc").read_text() == text
    assert '"v255"' not in text and "s_store" not in text and "s_dcache" not in text and "s_atomic" not in text
    assert {p.stem for p in CSRC.glob("d256_loop_*.inc")} == {f"d256_loop_{p.name}" for p in GEN.PROGRAMS}


def swizzled(row, chunk, rowbytes):
    chunks = rowbytes // 16
    return row * rowbytes + ((chunk ^ ((row // max(1, 256 // rowbytes)) & (chunks - 1))) << 4)


def walk(program, q, k, v, q_scale, k_scale, *, sm_scale, block, causal=False, bias=None, tiles=None, order=None):
    """What attention_d256_kernel hands to the program for one query block; (O, m, d) of its queries."""
    q_len, k_len = len(q), len(k)
    n_kb = -(-k_len // KEYS)
    padded = n_kb * KEYS
    memory = Memory()
    room = np.full((padded * DIM,), 0x5A, np.uint8)  # whatever lies behind the keys
    room[:k_len * DIM] = k.view(np.uint8).reshape(-1)
    k_base = memory.add(room)
    v_base = memory.add(pack_values(torch.from_numpy(v)).numpy())
    sums = v.reshape(DIM, n_kb, KEYS).astype(np.int64).sum(2).T * 128 + SEED_BITS
    sum_base, ks_base = memory.add(sums.astype(np.int32)), memory.add(k_scale)
    named = {"kptr": k_base, "vptr": v_base, "sumptr": sum_base, "ksptr": ks_base, "padded": padded,
             "qs2": int(np.float32(np.float32(sm_scale) * attention.LOG2E).view(np.uint32))}
    if program.listed:
        named["list"] = memory.add(np.asarray(tiles, np.int32))
        n_it = len(tiles)
    else:
        n_it = -(-min(k_len, (block + 1) * 128 if causal else k_len) // KEYS)
    if program.bias:
        named["mask"] = memory.add(bias)
    lds, waves = Lds(GEN.V_REGION + GEN.TILE_BYTES), []
    for wave in range(4):
        query = block * 128 + wave * 32 + L32
        ok = query < q_len
        rows = np.where(ok[:, None], q[np.minimum(query, q_len - 1)], 0).astype(np.int8)
        vector = {GEN.QSCALE: np.where(ok, q_scale[np.minimum(query // 16 * 8 + query % 8, len(q_scale) - 1)], np.float32(1)).view(np.uint32),
                  GEN.KA: GEN.K_REGION + np.array([swizzled(r, h, DIM) for r, h in zip(L32, HALF)]),
                  GEN.VA: GEN.V_REGION + np.array([swizzled(r, h, KEYS) for r, h in zip(L32, HALF)]),
                  GEN.KC: (LANE >> 4) * DIM + ((LANE & 15 ^ LANE >> 4) << 4),
                  GEN.VC: (LANE >> 3) * padded + ((LANE & 7 ^ LANE >> 4) << 4),
                  GEN.MRUN: np.full(64, np.float32(-50000)).view(np.uint32), GEN.DPART: 0}
        for kk in range(8):
            words = np.stack([rows[l, kk * 32 + HALF[l] * 16:][:16] for l in range(64)]).view(np.uint32)
            for at in range(4):
                vector[GEN.Q[kk] + at] = words[:, at]
        mine = dict(named, wave=wave, count=n_it - 1)
        mine["rem"] = 1 << 30 if program.bias else k_len - (n_it - 1) * KEYS
        mine["remq"] = block * 128 + wave * 32 + 1 - (n_it - 1) * KEYS if causal else 1 << 30
        waves.append(Wave(GEN.render(program), memory, lds, vector, mine))
    run_workgroup(waves, order)
    out, m, d = np.zeros((128, DIM), np.float32), np.zeros(128, np.float32), np.zeros(128, np.float32)
    for at, wave in enumerate(waves):
        for cb in range(8):
            for r in range(16):
                out[at * 32 + L32, cb * 32 + 8 * (r // 4) + 4 * HALF + r % 4] = wave.v[GEN.O[cb] + r].view(np.float32)
        m[at * 32 + L32] = wave.v[GEN.MRUN].view(np.float32)
        part = wave.v[GEN.DPART].view(np.float32)
        d[at * 32:at * 32 + 32] = part[:32] + part[32:]
    return out, m, d


CASES = [  # program, queries, keys, block, options
    ("raw", 128, 128, 0, {}), ("raw", 128, 300, 0, {}), ("raw", 250, 641, 1, {}), ("raw", 128, 65, 0, {}),
    ("scaled", 128, 384, 0, {"sm_scale": -0.05}), ("scaled", 128, 257, 0, {"sm_scale": 0.0}),
    ("scaled", 300, 300, 0, {"causal": True}), ("scaled", 300, 300, 2, {"causal": True}), ("scaled", 384, 150, 2, {"causal": True}),
    ("bias", 300, 300, 1, {"causal": True, "mask": "padding"}), ("bias", 300, 300, 2, {"causal": True, "mask": "float"}),
    ("bias_listed", 128, 700, 0, {"mask": "padding"}), ("bias_listed", 128, 700, 0, {"mask": "holes"}),
    ("bias_listed", 128, 640, 0, {"mask": "float"}), ("bias_listed", 100, 60, 0, {"mask": "float"}),
]


@pytest.mark.parametrize("name,q_len,k_len,block,options", CASES)
def test_walk_gives_the_oracles_output(name, q_len, k_len, block, options):
    random = np.random.default_rng(q_len + k_len + block)
    causal, kind, sm_scale = options.get("causal", False), options.get("mask"), options.get("sm_scale", 0.06)
    n_kb = -(-k_len // KEYS)
    padded = n_kb * KEYS
    q, k = (random.integers(-127, 128, (n, DIM)).astype(np.int8) for n in (q_len, k_len))
    v = np.zeros((DIM, padded), np.int8)
    v[:, :k_len] = random.integers(-127, 128, (DIM, k_len))
    q_scale = random.uniform(0.01, 0.03, -(-q_len // 128) * 64).astype(np.float32)
    k_scale = random.uniform(0.01, 0.03, n_kb * 4).astype(np.float32)
    mask = row = tiles = None
    if kind:
        mask = random.normal(size=k_len).astype(np.float32) if kind == "float" else random.random(k_len) < 2
        if kind == "padding":
            mask[k_len * 3 // 4:] = False
        elif kind == "holes":
            mask[128:384] = False
            mask[5::7] = False
        elif kind == "float":
            mask[::9] = -np.inf
        row = np.full(padded, -np.inf, np.float32)
        if mask.dtype == bool:
            row[:k_len] = np.where(mask, 0, -np.inf)
        else:
            row[:k_len] = mask * attention.LOG2E
        if name == "bias_listed":
            tiles = [t for t in range(n_kb) if np.isfinite(row[t * KEYS:(t + 1) * KEYS]).any()]
    listed = None
    if tiles is not None:
        listed = np.zeros((1, 1, n_kb + 1), np.int32)
        listed[0, 0, :len(tiles)], listed[0, 0, n_kb] = tiles, len(tiles)
    ones, zeros = np.ones(DIM, np.float32), np.zeros(DIM, np.float32)
    expected, lse, _ = attention.attend(
        q[None, None], k[None, None], v, q_scale[None, None], k_scale[None, None], ones, zeros, key_block=KEYS,
        sm_scale=sm_scale, mask=None if mask is None else mask[None, None, None], is_causal=causal, key_mask_tiles=listed,
        out_dtype="float16")
    first, last = block * 128, min(q_len, block * 128 + 128)
    results = [walk(PROGRAMS[name], q, k, v, q_scale, k_scale, sm_scale=sm_scale, block=block, causal=causal, bias=row,
                    tiles=tiles, order=order) for order in (None, (2, 0, 3, 1))]
    assert all(np.array_equal(a, b) for a, b in zip(*results))  # no race between the wavefronts of an interval
    out, m, d = (x[:last - first] for x in results[0])
    expected, lse = expected[0, 0, first:last], lse[0, 0, first:last]
    assert (d > 0).all()
    with np.errstate(divide="ignore"):
        # outputs are rounded to half precision (2^-11); exponentials are exact on both sides
        assert np.abs(out / d[:, None] - expected).max() <= 2.0 ** -11 * np.abs(expected).max()
        assert np.abs((np.log2(d) + m) / attention.LOG2E - lse).max() < 1e-4


def test_two_workgroups_share_a_compute_unit():
    """(registers of a SIMD: 512 for two wavefronts; LDS: 160 KB for two workgroups)"""
    from risaattention_amd import native
    from tests.test_kernel_registers import code_objects, kernels, workgroups

    found = [k for elf in code_objects(native.library_path().read_bytes()) for k in kernels(elf) if "attention_d256_kernel" in k[".name"]]
    assert len(found) == len(GEN.PROGRAMS)
    for kernel in found:
        assert workgroups(kernel) == 2 and kernel[".private_segment_fixed_size"] == 0
        assert kernel[".sgpr_spill_count"] == kernel[".vgpr_spill_count"] == 0
    assert 2 * (GEN.V_REGION + GEN.TILE_BYTES) <= 160 * 1024
