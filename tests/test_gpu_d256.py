"""Head dim 256 with thirty-two queries per wavefront (launches of more workgroups than compute units)
against the sixteen-query kernel (RISA_COMPILED_LOOP=1), which adds a row's denominator up in another
order, and the oracle: key ranges at the edges of tiles, ragged query blocks, every mode."""

import math

import pytest
import torch

from tests.helpers import oracle_prequantize, relative_l2, seeded, to_numpy
from tests.test_gpu_tile_loop import compiled_loop

pytestmark = pytest.mark.gpu


def both(risa, q, k, v, **options):
    mine, lse = risa.int8_attention(q, k, v, return_lse=True, **options)
    with compiled_loop():
        theirs, their_lse = risa.int8_attention(q, k, v, return_lse=True, **options)
    # denominators differ by FP32 rounding, a bfloat16 output by one step (2^-8) where that crosses
    # a rounding boundary: one value in some thousands
    assert relative_l2(to_numpy(mine), to_numpy(theirs)) < 2e-4
    assert torch.equal(torch.isfinite(lse), torch.isfinite(their_lse))
    seen = torch.isfinite(lse)
    assert (lse - their_lse)[seen].abs().max() < 1e-4
    return mine


@pytest.mark.parametrize("k_len", [1025, 1152, 1279, 1281, 2048])
@pytest.mark.parametrize("q_len,heads", [(513, 104), (128, 514), (100, 513)])
@pytest.mark.parametrize("mode", ["raw", "negative", "causal", "padding", "bias", "bias_causal"])
def test_modes(risa, mode, q_len, heads, k_len):
    q = seeded((1, heads, q_len, 256), torch.bfloat16, q_len, scale=1.5)
    k = seeded((1, 1, k_len, 256), torch.bfloat16, k_len + 1, scale=1.5)
    v = seeded((1, 1, k_len, 256), torch.bfloat16, k_len + 2, offset=0.25)
    options = {"is_causal": mode.endswith("causal")}
    if mode == "negative":
        options["scale"] = -0.05
    elif mode == "padding":
        options["attn_mask"] = (torch.arange(k_len, device="cuda") < k_len * 2 // 3)[None, None, None]
    elif mode.startswith("bias"):
        mask = seeded((1, 1, 1, k_len), torch.float32, k_len)
        mask[..., ::97] = -math.inf
        mask[..., 256:384] = -math.inf  # a hidden tile
        mask[..., 384:512] = -0.0
        options["attn_mask"] = mask
    out = both(risa, q, k, v, **options)
    if mode in ("raw", "bias") and heads == 514 and k_len == 1281:
        from oracle import pipeline

        prepared = oracle_prequantize(q[:, :1], k, v, return_lse=True, **options)
        expected, _, _ = pipeline.attend(prepared, return_lse=True)
        assert relative_l2(to_numpy(out[:, :1]), expected) < 1e-3


@pytest.mark.parametrize("masked", [False, True])
def test_rows_that_see_no_key(risa, masked):
    q = seeded((1, 514, 128, 256), torch.float16, 3)
    k, v = seeded((1, 1, 1300, 256), torch.float16, 4), seeded((1, 1, 1300, 256), torch.float16, 5)
    mask = torch.zeros(1, 1, 1, 1300, dtype=torch.bool, device="cuda")
    if masked:
        mask[..., 700:] = True  # rows below see nothing under the causal rule
    out, lse = risa.int8_attention(q, k, v, attn_mask=mask, is_causal=masked, return_lse=True)
    assert not out.any() and torch.isneginf(lse).all()


@pytest.mark.parametrize("dim,token_major", [(256, False), (200, True)])
@pytest.mark.parametrize("mode", ["raw", "causal", "padding", "padding_causal", "rows", "rows_causal", "head_rows"])
def test_every_batch_head_and_mask_plane(risa, mode, dim, token_major):
    """Grouped heads over several batches: masks of another length per batch, additive rows per (batch, head) and
    per head, tile lists of their own, both layouts, rows that the preparation pads."""
    batch, heads, kv_heads, causal = 2, 36, 12, mode.endswith("causal")
    q_len, k_len = (1100, 1181) if causal else (650, 1281)

    def tensor(count, length, seed, **options):
        if token_major:
            return seeded((batch, length, count, dim), torch.bfloat16, seed, **options).transpose(1, 2)
        return seeded((batch, count, length, dim), torch.bfloat16, seed, **options)

    q, k = tensor(heads, q_len, 1, scale=1.5), tensor(kv_heads, k_len, 2, scale=1.5)
    v = tensor(kv_heads, k_len, 3, offset=0.25)
    mask = None
    if mode.startswith("padding"):
        mask = torch.arange(k_len, device="cuda") < torch.tensor([k_len, 700], device="cuda")[:, None, None, None]
    elif "rows" in mode:
        mask = seeded((1 if mode == "head_rows" else batch, heads, 1, k_len), torch.float32, 4)
        mask[..., ::97] = -math.inf
        mask[:, ::2, :, 256:512] = -math.inf  # tiles hidden from every other head
    options = {"attn_mask": mask, "is_causal": causal}
    out = both(risa, q, k, v, **options)
    packed = risa.prequantize_int8_attention(q, k, v, **options)
    rows = risa.int8_attention_from_prequantized(packed, output_layout="nhd")
    assert rows.stride(1) < rows.stride(2) and torch.equal(rows, out)

    from oracle import pipeline

    of_last = None if mask is None else mask[-1:, -1:]
    prepared = oracle_prequantize(q[-1:, -1:], k[-1:, -1:], v[-1:, -1:], attn_mask=of_last, is_causal=causal, return_lse=True)
    expected, _, _ = pipeline.attend(prepared, return_lse=True)
    assert relative_l2(to_numpy(out[-1:, -1:]), expected) < 1e-3
