"""Registers of the built attention kernels, read from the metadata the compiler leaves beside them.
A wavefront's registers decide how many workgroups share a compute unit, and a kernel one register
above a limit loses one of them without any other sign."""

import re
import struct

import msgpack
import pytest

from risaattention_amd import native

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
SCALAR, VECTOR, STAGED, LANES = range(4)  # attention_kernel's MASK_MODE
BOOL, KEY_BIAS, FLOATS = 3, 4, (0, 1, 2)  # its MASK_DT


def code_objects(data):
    for match in re.finditer(re.escape(BUNDLE), data):
        at = match.start() + len(BUNDLE)
        (entries,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            if b"gfx950" in data[at + 24:at + 24 + length]:
                yield data[match.start() + offset:match.start() + offset + size]
            at += 24 + length


def kernels(elf):
    """Metadata of every kernel of one code object (a note of owner AMDGPU, type 32)."""
    note = re.search(rb"\x07\0\0\0(....)\x20\0\0\0AMDGPU\0\0", elf, re.S)
    (size,) = struct.unpack("<I", note.group(1))
    return msgpack.unpackb(elf[note.end():note.end() + size])["amdhsa.kernels"]


def variants(template):
    """Template arguments -> metadata."""
    found = {}
    for elf in code_objects(native.library_path().read_bytes()):
        for kernel in kernels(elf):
            name = re.search(template + r"I((?:L[ib]n?\d+E)+)E", kernel[".name"])
            if name:
                found[tuple(int(x.replace("n", "-")) for x in re.findall(r"L[ib](n?\d+)E", name.group(1)))] = kernel
    return found


@pytest.fixture(scope="module")
def attention_kernels():
    """(D, CTA_K, FAST, INDEXED, CAPTURE, MASK_DT, MASK_MODE) -> metadata."""
    found = variants("16attention_kernel")
    assert len(found) > 50
    return found


def workgroups(kernel):
    """Per compute unit: one wavefront on each of four SIMDs, 512 registers there, handed out by
    eights (the count holds the accumulation registers too)."""
    return 512 // (-(-kernel[".vgpr_count"] // 8) * 8)


def test_lane_words_of_head_dim_64_leave_room_for_four_workgroups(attention_kernels):
    for indexed, capture in ((0, 0), (1, 0), (0, 1)):
        assert workgroups(attention_kernels[64, 64, 0, indexed, capture, BOOL, LANES]) == 4, (indexed, capture)
    assert attention_kernels[64, 64, 0, 1, 0, BOOL, LANES][".private_segment_fixed_size"] == 0


def test_hand_scheduled_loops_of_head_dim_64_leave_room_for_three_workgroups(attention_kernels):
    for fast, indexed, mask in ((1, 0, -1), (0, 0, -1), (0, 0, KEY_BIAS), (0, 1, KEY_BIAS)):
        kernel = attention_kernels[64, 64, fast, indexed, 0, mask, SCALAR]
        assert workgroups(kernel) == 3 and kernel[".private_segment_fixed_size"] == 0, (fast, indexed, mask)


def test_float_masks_read_per_score_leave_room_for_three_workgroups(attention_kernels):
    for mask in FLOATS:
        for indexed in (0, 1):
            kernel = attention_kernels[64, 64, 0, indexed, 0, mask, SCALAR]
            assert workgroups(kernel) == 3 and kernel[".private_segment_fixed_size"] == 0, (mask, indexed)


def test_key_only_masks_spill_no_scalar_register(attention_kernels):
    """Spilled around the hand-scheduled loop, sixteen of them cost launches of one or two key tiles 2-6 %."""
    for shape in ((64, 64), (128, 128)):
        for indexed in (0, 1):
            assert attention_kernels[(*shape, 0, indexed, 0, KEY_BIAS, SCALAR)][".sgpr_spill_count"] == 0, (shape, indexed)


def test_ranges_of_the_keys_are_kernels_of_their_own():
    """Their run-time tests would take scalar registers and instructions from every walk over all tiles."""
    narrow = variants("23attention_narrow_kernel")  # (..., RANGES)
    ranges = {arguments[:-1] for arguments in narrow if len(arguments) == 10 and arguments[-1]}
    assert len(ranges) == 60 and all((*arguments, 0) in narrow for arguments in ranges)
