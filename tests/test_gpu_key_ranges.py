"""Launches of few query blocks, whose key tiles workgroups of their own walk in ranges, against the walk
of all tiles by one workgroup (no workspace for partial results): only the order of FP32 additions
differs.  Ragged lengths, more ranges than tiles in a list, rows that see nothing, every mask form."""

import math

import pytest
import torch

from risaattention_amd import attend
from tests.helpers import oracle_prequantize, relative_l2, seeded, to_numpy

pytestmark = pytest.mark.gpu


def mask_for(kind, q_len, k_len):
    if kind in ("plain", "negative", "causal"):
        return None
    pick = torch.Generator(device="cuda").manual_seed(q_len + k_len)
    if kind.startswith("padding"):
        return (torch.arange(k_len, device="cuda") < k_len * 3 // 5)[None, None, None]
    if kind == "one_tile":  # a list of one tile under several ranges
        mask = torch.zeros(1, 1, 1, k_len, dtype=torch.bool, device="cuda")
        mask[..., k_len // 2] = True
        return mask
    if kind == "key_bias":
        mask = torch.randn(1, 1, 1, k_len, generator=pick, device="cuda")
        mask[..., ::7] = -math.inf
        return mask
    if kind == "bool":
        mask = torch.rand(1, 1, q_len, k_len, generator=pick, device="cuda") < 0.5
        mask[:, :, 3:9] = False
        mask[:, :, 9:12, : k_len - 5] = False  # only the last range sees a key
        return mask
    mask = torch.randn(1, 1, q_len, k_len, generator=pick, device="cuda")
    mask[torch.rand(mask.shape, generator=pick, device="cuda") < 0.1] = -math.inf
    mask[:, :, 3:9] = -math.inf
    mask[:, :, 20:24, ::3] = torch.finfo(torch.float32).min
    mask[:, :, 20:24, 1::3] = math.nan
    return mask.to(getattr(torch, kind))


@pytest.mark.parametrize("dim", [64, 128, 256, 80])
@pytest.mark.parametrize("q_len,k_len,heads", [(257, 2500, 4), (1, 4099, 8), (1500, 1500, 2), (33, 1024, 2)])
@pytest.mark.parametrize("kind", ["plain", "negative", "causal", "padding", "padding_causal", "one_tile", "key_bias", "bool", "float32", "bfloat16"])
def test_ranges_of_the_keys(risa, monkeypatch, kind, q_len, k_len, heads, dim):
    q = seeded((1, heads, q_len, dim), torch.bfloat16, q_len, scale=1.5)
    k = seeded((1, 1, k_len, dim), torch.bfloat16, k_len + 1, scale=1.5)
    v = seeded((1, 1, k_len, dim), torch.bfloat16, k_len + 2, offset=0.25)
    options = {"attn_mask": mask_for(kind, q_len, k_len), "is_causal": kind.endswith("causal")}
    if kind == "negative":
        options["scale"] = -0.05
    packed = risa.prequantize_int8_attention(q, k, v, return_lse=True, **options)
    sizes = []
    with monkeypatch.context() as patch:
        patch.setattr(attend, "attention_split_bytes", lambda *extents: sizes.append(extents) or 0)
        whole, whole_lse = risa.int8_attention_from_prequantized(packed, return_lse=True)
    out, lse = risa.int8_attention_from_prequantized(packed, return_lse=True)
    if k_len > 2000:
        assert attend.attention_split_bytes(*sizes[0]) > 0
    # (a bfloat16 output moves by one step where FP32 rounding crosses a boundary)
    assert relative_l2(to_numpy(out), to_numpy(whole)) < 2e-4
    seen = torch.isfinite(lse)
    assert torch.equal(seen, torch.isfinite(whole_lse))
    assert not seen.any() or (lse - whole_lse)[seen].abs().max() < 1e-4
    assert torch.equal(out, risa.int8_attention(q, k, v, **options))
    if kind in ("plain", "bool") and (q_len, dim) == (257, 128):
        from oracle import pipeline

        prepared = oracle_prequantize(q, k, v, return_lse=True, **options)
        expected, _, _ = pipeline.attend(prepared, return_lse=True)
        assert relative_l2(to_numpy(out), expected) < 1e-3


def test_captured_into_a_graph(risa):
    q, k, v = (seeded((1, 2, n, 128), torch.bfloat16, n) for n in (200, 3000, 3000))
    expected = risa.int8_attention(q, k, v)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = risa.int8_attention(q, k, v)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, expected)
        risa.int8_attention(k, q, q)  # eager work between the replays
        out.zero_()
