"""Log-normalisers from one native call against the packed route: the same bits.

The packed route adds the anchor correction to the log-normalisers as tensors; the single call stores
it first and lets the attention kernel add its term.  Both are one FP32 addition, so results are equal
bit for bit in every form the call takes: kernels of few and of many workgroups, split key ranges, rows
that the preparation pads, every mask form, types and layouts.
"""

from __future__ import annotations

import pytest
import torch

import risaattention_amd as risa

pytestmark = pytest.mark.gpu

FORMS = [
    # batch, q_heads, kv_heads, q_len, k_len, dim, dtype, mode, causal, mask, token-major
    (1, 2, 1, 1, 65, 64, torch.bfloat16, "absmax", False, None, False),
    (1, 4, 2, 129, 300, 80, torch.float16, "midpoint_affine", False, None, True),
    (2, 4, 4, 65, 257, 40, torch.float32, "absmax", True, None, False),
    (1, 3, 1, 77, 1500, 39, torch.bfloat16, "absmax", False, "padding", False),
    (1, 16, 4, 2048, 2100, 128, torch.bfloat16, "absmax", False, None, False),
    (2, 24, 24, 1000, 1300, 64, torch.bfloat16, "absmax", False, "bool", False),
    (2, 24, 8, 1000, 1300, 128, torch.float16, "midpoint_affine", False, "padding", True),
    (1, 40, 8, 1025, 900, 128, torch.float32, "absmax", False, "bias", False),
    (1, 40, 8, 1100, 1100, 200, torch.bfloat16, "absmax", True, None, False),
    (1, 24, 8, 1500, 1280, 256, torch.bfloat16, "absmax", False, None, False),
    # head dim 256 with a ragged last key tile and more workgroups than compute units (two under the causal rule)
    (2, 24, 8, 1500, 1025, 256, torch.bfloat16, "absmax", False, None, False),
    (1, 24, 8, 1500, 1999, 200, torch.float16, "midpoint_affine", False, "key_bias", True),
    (2, 24, 8, 1500, 1333, 256, torch.bfloat16, "absmax", False, "padding", False),
    (2, 24, 8, 1500, 1500, 256, torch.bfloat16, "absmax", True, None, False),
    (1, 16, 16, 128, 4096, 128, torch.bfloat16, "absmax", False, "padding", False),  # split key ranges
    # mask forms made by workgroups of the preparation: one launch and two, lane words of aligned rows
    # (the packed route makes all of them in launches of their own)
    (2, 24, 24, 1000, 1296, 64, torch.bfloat16, "absmax", False, "bool", False),
    (3, 16, 16, 1153, 4160, 128, torch.bfloat16, "midpoint_affine", False, "bool", False),
    (2, 24, 24, 512, 512, 64, torch.float16, "absmax", False, "bool", False),
    (1, 40, 8, 1025, 6016, 80, torch.bfloat16, "absmax", False, "documents", False),
    (2, 8, 8, 256, 512, 64, torch.bfloat16, "absmax", False, "padding", False),
    (2, 24, 24, 260, 1025, 64, torch.float32, "absmax", False, "key_bias", False),
    (1, 24, 8, 1000, 5000, 256, torch.bfloat16, "midpoint_affine", True, "key_bias", False),
]


@pytest.mark.parametrize("form", FORMS, ids=lambda f: "-".join(str(v).replace("torch.", "") for v in f))
def test_one_call_matches_packed_route(form):
    batch, q_heads, kv_heads, q_len, k_len, dim, dtype, mode, causal, mask_kind, token_major = form
    generator = torch.Generator().manual_seed(q_len + k_len + dim)

    def rows(heads, length):
        if token_major:
            return torch.randn(batch, length, heads, dim, generator=generator).to(dtype).cuda().transpose(1, 2)
        return torch.randn(batch, heads, length, dim, generator=generator).to(dtype).cuda()

    q, k, v = rows(q_heads, q_len), rows(kv_heads, k_len), rows(kv_heads, k_len)
    k += 3.0  # keys off the origin: an anchor is taken off
    mask = None
    if mask_kind == "padding":
        mask = (torch.arange(k_len) < k_len * 3 // 4)[None, None, None].cuda()
    elif mask_kind == "bool":
        mask = torch.rand(batch, 1, q_len, k_len, generator=generator) < 0.7
        mask[:, :, :5] = False  # rows that see no key
        mask = mask.cuda()
    elif mask_kind == "documents":
        mask = (torch.arange(q_len)[:, None] * 8 // q_len == torch.arange(k_len) * 8 // k_len)[None, None].cuda()
    elif mask_kind == "key_bias":
        mask = torch.randn(batch, 1, 1, k_len, generator=generator)
        mask[:, :, :, 128:400] = -torch.inf
        mask = mask.half().cuda()
    elif mask_kind == "bias":
        mask = torch.randn(batch, 1, q_len, k_len, generator=generator).cuda()
    packed = risa.prequantize_int8_attention(q, k, v, attn_mask=mask, v_quantization=mode, is_causal=causal,
                                             return_lse=True)
    expected, expected_lse = risa.int8_attention_from_prequantized(packed, return_lse=True)
    out, lse = risa.int8_attention(q, k, v, attn_mask=mask, v_quantization=mode, is_causal=causal, return_lse=True)
    torch.cuda.synchronize()
    assert out.dtype == expected.dtype and lse.dtype == torch.float32 and lse.is_contiguous()
    assert torch.equal(out, expected)
    assert torch.equal(lse, expected_lse)
    assert bool((packed.lse_shift != 0).any())
