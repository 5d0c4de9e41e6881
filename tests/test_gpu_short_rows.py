"""Rows of fewer channels than the kernel's head dim, read in place by the preparation kernels,
against the same values padded with zeros beforehand (what rows off a 16-byte boundary, or of a
channel count that is no multiple of eight, still go through): bit for bit, every prepared tensor
and the output, on each launch shape of the preparation."""

import pytest
import torch

from risaattention_amd.prepare import rows_hold_whole_runs
from tests.helpers import oracle_prequantize, seeded, to_numpy

pytestmark = pytest.mark.gpu


def off_boundary(tensor):
    """The same values in rows that start off a 16-byte boundary."""
    wide = torch.full((*tensor.shape[:-1], tensor.shape[-1] + 9), float("nan"), dtype=tensor.dtype, device=tensor.device)
    wide[..., 1:-8] = tensor
    return wide[..., 1:-8]


@pytest.mark.parametrize("dim", [8, 40, 72, 80, 120, 136, 200, 248])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("mode", ["absmax", "midpoint_affine"])
@pytest.mark.parametrize("q_len,k_len,kv_heads", [(1, 1, 1), (130, 200, 2), (300, 1025, 2), (90, 4097, 1), (4200, 4300, 2)])
def test_equal_padded_rows(risa, dim, dtype, mode, q_len, k_len, kv_heads):
    q = seeded((2, 2 * kv_heads, q_len, dim), dtype, dim, scale=2.0)
    k = seeded((2, kv_heads, k_len, dim), dtype, dim + 1, offset=0.5)
    v = seeded((2, kv_heads, k_len, dim), dtype, dim + 2, offset=-0.25)
    # token-major storage and, at the very end of it, the last row of the last head
    nhd = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
    assert rows_hold_whole_runs(*nhd) and not rows_hold_whole_runs(*map(off_boundary, (q, k, v)))
    for mine in ((q, k, v), nhd):
        packed = risa.prequantize_int8_attention(*mine, v_quantization=mode)
        padded = risa.prequantize_int8_attention(*map(off_boundary, mine), v_quantization=mode)
        for name in ("q", "k", "v", "q_scale", "k_scale", "v_scale", "v_center", "v_tile_sum"):
            assert torch.equal(getattr(packed, name), getattr(padded, name)), name
        out = risa.int8_attention(*mine, v_quantization=mode)
        assert torch.equal(out, risa.int8_attention(*map(off_boundary, mine), v_quantization=mode))
    if k_len <= 300:
        expected = oracle_prequantize(q, k, v, v_quantization=mode)
        assert (packed.q.cpu().numpy() == expected.q).all() and (packed.k.cpu().numpy() == expected.k).all()
        assert (to_numpy(packed.v_center) == expected.v_center).all()


def test_gathered_keys_and_channel_counts(risa):
    q, k, v = (seeded((1, 2, 700, 80), torch.bfloat16, i) for i in range(3))
    order = torch.randperm(700, generator=torch.Generator().manual_seed(0)).cuda()
    order = risa.prepare_kv_permutation(order.to(torch.int32).expand(1, 2, 700).contiguous())
    mine = risa.int8_attention(q, k, v, kv_permutation=order)
    assert torch.equal(mine, risa.int8_attention(*map(off_boundary, (q, k, v)), kv_permutation=order))
    for dim in (1, 12, 100, 255):  # no whole runs of eight: padded beforehand
        odd = [seeded((1, 2, 65, dim), torch.bfloat16, i) for i in range(3)]
        assert not rows_hold_whole_runs(*odd)
        assert torch.isfinite(risa.int8_attention(*odd)).all()
