"""Launches of few query blocks, whose key tiles workgroups of their own walk in ranges, against the walk
of all tiles by one workgroup (no workspace for partial results): only the order of FP32 additions
differs.  Ragged lengths, more ranges than tiles in a list, rows that see nothing, every mask form."""

import math

import pytest
import torch

from risaattention_amd import attend
from tests.helpers import oracle_prequantize, relative_l2, seeded, to_numpy

pytestmark = pytest.mark.gpu


def mask_for(kind, batch, heads, q_len, k_len):
    if kind in ("plain", "negative", "causal"):
        return None
    pick = torch.Generator(device="cuda").manual_seed(q_len + k_len)
    if kind.startswith("padding"):  # another length per batch
        lengths = torch.tensor([k_len * 3 // 5, k_len * 4 // 5][:batch], device="cuda")
        return (torch.arange(k_len, device="cuda") < lengths[:, None])[:, None, None]
    if kind == "one_tile":  # a list of one tile under several ranges
        mask = torch.zeros(1, 1, 1, k_len, dtype=torch.bool, device="cuda")
        mask[..., k_len // 2] = True
        return mask
    if kind == "key_bias":  # another row per head
        mask = torch.randn(1, heads, 1, k_len, generator=pick, device="cuda")
        mask[..., ::7] = -math.inf
        return mask
    if kind == "bool":
        mask = torch.rand(batch, 1, q_len, k_len, generator=pick, device="cuda") < 0.5
        mask[:, :, 3:9] = False
        mask[:, :, 9:12, : k_len - 5] = False  # only the last range sees a key
        return mask
    mask = torch.randn(1, heads, q_len, k_len, generator=pick, device="cuda")
    mask[torch.rand(mask.shape, generator=pick, device="cuda") < 0.1] = -math.inf
    mask[:, :, 3:9] = -math.inf
    mask[:, :, 20:24, ::3] = torch.finfo(torch.float32).min
    mask[:, :, 20:24, 1::3] = math.nan
    return mask.to(getattr(torch, kind))


KINDS = ["plain", "negative", "padding", "one_tile", "key_bias", "bool", "float32", "bfloat16"]
SHAPES = [(1, 4, 1, 257, 2500), (1, 8, 1, 1, 4099), (1, 4, 4, 33, 3000), (2, 4, 2, 257, 2500)]
# (a query block's keys end with its queries, so the ranges are those of long query rows)
CAUSAL_SHAPES = [(1, 2, 1, 3000, 2700), (2, 4, 2, 1300, 2600), (1, 2, 2, 4099, 4099)]


@pytest.mark.parametrize("dim", [64, 128, 256, 80])
@pytest.mark.parametrize("kind,shape", [(kind, shape) for kind in KINDS for shape in SHAPES] +
                         [(kind, shape) for kind in ("causal", "padding_causal") for shape in CAUSAL_SHAPES])
def test_ranges_of_the_keys(risa, monkeypatch, kind, shape, dim):
    batch, heads, kv_heads, q_len, k_len = shape
    q = seeded((batch, heads, q_len, dim), torch.bfloat16, q_len, scale=1.5)
    k = seeded((batch, kv_heads, k_len, dim), torch.bfloat16, k_len + 1, scale=1.5)
    v = seeded((batch, kv_heads, k_len, dim), torch.bfloat16, k_len + 2, offset=0.25)
    options = {"attn_mask": mask_for(kind, batch, heads, q_len, k_len), "is_causal": kind.endswith("causal")}
    if kind == "negative":
        options["scale"] = -0.05
    packed = risa.prequantize_int8_attention(q, k, v, return_lse=True, **options)
    calls = []
    with monkeypatch.context() as patch:
        patch.setattr(attend, "attention_split_bytes", lambda *call: calls.append(call) or 0)
        whole, whole_lse = risa.int8_attention_from_prequantized(packed, return_lse=True)
    out, lse = risa.int8_attention_from_prequantized(packed, return_lse=True)
    assert attend.attention_split_bytes(*calls[0]) > 0  # the size of this call: it is split
    # (a bfloat16 output moves by one step where FP32 rounding crosses a boundary)
    assert relative_l2(to_numpy(out), to_numpy(whole)) < 2e-4
    seen = torch.isfinite(lse)
    assert torch.equal(seen, torch.isfinite(whole_lse))
    assert not seen.any() or (lse - whole_lse)[seen].abs().max() < 1e-4
    assert torch.equal(out, risa.int8_attention(q, k, v, **options))
    if kind in ("plain", "bool") and (batch, q_len, dim) == (1, 257, 128):
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
