"""The tile loops of gen_tile_loops.py against the loop the compiler schedules
(RISA_COMPILED_LOOP=1), bit for bit, on launches of more workgroups than compute units: causal
launches, scales of both signs, short key ranges and masks, at the edges of tiles and query blocks."""

import math

import pytest
import torch

from tests.helpers import oracle_prequantize, relative_l2, seeded, to_numpy
from tests.test_gpu_tile_loop import compiled_loop

pytestmark = pytest.mark.gpu


def both(risa, *tensors, **options):
    """Through packed operands (log-normalisers asked for: no room behind the keys below 2048, so a
    last tile of fewer keys leaves two tiles to the compiled loop) and in one call (V codes behind the
    keys: the loop copies such a tile whole)."""
    mine = risa.int8_attention(*tensors, return_lse=True, **options)
    one_call = risa.int8_attention(*tensors, **options)
    with compiled_loop():
        theirs = risa.int8_attention(*tensors, return_lse=True, **options)
    for a, b in zip((*mine, one_call), (*theirs, theirs[0])):
        # (rows that see nothing but infinite terms are no numbers on both sides)
        assert torch.equal(torch.nan_to_num(a.float(), nan=123.0), torch.nan_to_num(b.float(), nan=123.0))
    return mine


def inputs(batch, heads, kv_heads, q_len, k_len, dim, dtype=torch.bfloat16, scale=1.5):
    return (seeded((batch, heads, q_len, dim), dtype, q_len, scale=scale),
            seeded((batch, kv_heads, k_len, dim), dtype, k_len + 1, scale=scale),
            seeded((batch, kv_heads, k_len, dim), dtype, k_len + 2, offset=0.25))


@pytest.mark.parametrize("q_len,k_len", [(1152, 1152), (1153, 1153), (2000, 2000), (2304, 1300), (1200, 2304), (600, 600), (513, 513), (2500, 2300)])
@pytest.mark.parametrize("dim", [128, 64])
def test_causal(risa, dim, q_len, k_len):
    q, k, v = inputs(1, 60, 4, q_len, k_len, dim)
    out, lse = both(risa, q, k, v, is_causal=True)
    from oracle import pipeline

    prepared = oracle_prequantize(q[:, :1], k[:, :1], v[:, :1], return_lse=True, is_causal=True)
    expected, _, _ = pipeline.attend(prepared, return_lse=True)
    assert relative_l2(to_numpy(out[:, :1]), expected) < 1e-3


@pytest.mark.parametrize("k_len", [65, 128, 129, 512, 511, 1024, 1025, 1216, 2048])
@pytest.mark.parametrize("scale", [None, -0.1, 0.0])
@pytest.mark.parametrize("dim", [128, 64])
def test_key_range_and_scale(risa, dim, scale, k_len):
    q, k, v = inputs(2, 20, 4, 1030, k_len, dim, torch.float16)
    both(risa, q, k, v, scale=scale)


@pytest.mark.parametrize("q_len,k_len", [(1024, 1024), (1030, 512), (1152, 1100), (1153, 64), (896, 200), (1024, 128)])
@pytest.mark.parametrize("kind", ["f32", "f32_no_inf", "bf16", "bool", "bool_head"])
@pytest.mark.parametrize("dim", [128, 64])
def test_query_masks(risa, dim, kind, q_len, k_len):
    """Float masks with hidden keys, numbers at the ends of the range, infinities and NaN, rows that
    see nothing; boolean masks shared by the heads and per head; with and without the causal rule."""
    q, k, v = inputs(2, 20, 4, q_len, k_len, dim)
    pick = torch.Generator(device="cuda").manual_seed(q_len + k_len)
    if kind.startswith("bool"):
        mask = torch.rand(2, 20 if kind == "bool_head" else 1, q_len, k_len, generator=pick, device="cuda") < 0.7
        mask[:, :, 5:9] = False
        mask[:, :, :, : k_len // 2] |= torch.arange(q_len, device="cuda")[:, None] % 3 == 0
    else:
        mask = torch.randn(2, 1, q_len, k_len, generator=pick, device="cuda")
        chance = torch.rand(mask.shape, generator=pick, device="cuda")
        for low, term in ((0.90, -math.inf), (0.98, torch.finfo(torch.float32).min), (0.99, math.inf), (0.995, math.nan)):
            if kind == "f32_no_inf" and term == math.inf:
                term = math.nan
            mask[(chance > low) & (torch.arange(q_len, device="cuda")[:, None] % 2 == 0)] = term
        mask[:, :, 5:9] = -math.inf
        mask = mask.to(torch.bfloat16 if kind == "bf16" else torch.float32)
    both(risa, q, k, v, attn_mask=mask)
    if q_len >= k_len:
        both(risa, q, k, v, attn_mask=mask, is_causal=True)


@pytest.mark.parametrize("q_len,k_len,pitch", [(1024, 512, 520), (1152, 200, 1204), (1030, 1090, 1092)])
@pytest.mark.parametrize("dim", [128, 64])
def test_float_mask_rows_of_a_wider_tensor(risa, dim, q_len, k_len, pitch):
    q, k, v = inputs(2, 20, 4, q_len, k_len, dim)
    wide = seeded((2, 1, q_len, pitch), torch.float32, q_len)
    wide[..., k_len:] = math.nan
    out, _ = both(risa, q, k, v, attn_mask=wide[..., :k_len])
    assert torch.equal(out, risa.int8_attention(q, k, v, attn_mask=wide[..., :k_len].contiguous()))


@pytest.mark.parametrize("k_len", [100, 1024, 1025, 1290, 2304, 2300])
@pytest.mark.parametrize("kind", ["padding", "bias", "sparse_bias"])
@pytest.mark.parametrize("dim", [128, 64])
def test_key_masks(risa, dim, kind, k_len):
    q, k, v = inputs(2, 20, 4, 1100, k_len, dim)
    if kind == "padding":
        mask = (torch.arange(k_len, device="cuda") < torch.tensor([[k_len], [k_len * 2 // 3]], device="cuda"))[:, None, None]
    else:
        mask = seeded((2, 1, 1, k_len), torch.float32, k_len)
        if kind == "sparse_bias":  # tiles of zeros, of both signs, among others, and hidden keys
            mask = torch.where(torch.arange(k_len, device="cuda") // 64 % 3 == 1, mask, mask * -0.0)
            mask[..., ::97] = -math.inf
    both(risa, q, k, v, attn_mask=mask)
    both(risa, q, k, v, attn_mask=mask.expand(2, 20, 1, k_len).contiguous(), is_causal=k_len <= 1100)


@pytest.mark.parametrize("k_len", [2049, 2300, 4223])
def test_key_codes_without_room_behind_them(risa, k_len):
    """Packed keys in storage of their own size (a saved or copied container): the last tile of fewer
    keys is then copied key by key; the results are those of the container with room behind."""
    import dataclasses

    q, k, v = inputs(1, 40, 4, 1045, k_len, 128)
    packed = risa.prequantize_int8_attention(q, k, v, return_lse=True)
    assert packed.k.is_contiguous() and packed.k.untyped_storage().nbytes() >= packed.k.numel() + packed.cta_k * 128
    exact = dataclasses.replace(packed, k=packed.k.clone())
    assert exact.k.untyped_storage().nbytes() < packed.k.untyped_storage().nbytes()
    for a, b in zip(risa.int8_attention_from_prequantized(packed, return_lse=True),
                    risa.int8_attention_from_prequantized(exact, return_lse=True)):
        assert torch.equal(a, b)
