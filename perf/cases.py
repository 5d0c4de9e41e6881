"""The attention calls whose speed matters to users of this package, over the range they are made in.

Every case is one call through the public entry points (`int8_attention`,
`construct_sparse_int8_attention`, `sparse_int8_attention`, or `prequantize_int8_attention`
followed by `int8_attention_from_prequantized`), preparation of Q, K and V included, as a model's
forward pass makes it.  The lengths, head counts and masks are those of the package's own
benchmark, tests and ComfyUI adapter.
"""

import math

import torch

import risaattention_amd as risa

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

DEFAULTS = {
    "path": "dense",        # dense | construct | reuse | split
    "batch": 1, "q_heads": 16, "kv_heads": 4, "q_len": 1024, "k_len": 1024, "dim": 128,
    "dtype": "bf16", "mode": "absmax", "causal": False, "lse": False,
    "mask": "none",         # none | key_padding | key_bias | bool | bias | documents | window
    "mask_dtype": "bool",   # element type of the additive masks
    "nhd": False,           # inputs stored token-major (a projection's output, seen head-major)
    "inputs": "normal",     # normal | outliers | blocks
}


def _case(**values):
    return {**DEFAULTS, **values}


def listed():
    return [
        # The shortest row of the package's throughput table: launches and host work count.
        _case(name="dense_512", q_len=512, k_len=512),
        # A middle row of the same table in the other value mode.
        _case(name="dense_2k_affine", q_len=2048, k_len=2048, mode="midpoint_affine"),
        # The headline row: one long sequence, grouped heads.
        _case(name="dense_32k", q_len=32768, k_len=32768),
        # Prefill of a decoder: grouped heads under the causal rule.
        _case(name="causal_8k", q_heads=32, kv_heads=8, q_len=8192, k_len=8192, causal=True),
        # Self-attention of an image model: a head dim the kernels pad, half precision, the
        # conditional and unconditional branch as a batch, projections stored token-major.
        _case(name="image_4k_dim80", batch=2, q_heads=8, kv_heads=8, q_len=4096, k_len=4096, dim=80,
              dtype="fp16", nhd=True),
        # The widest head dim.
        _case(name="wide_heads_8k", q_len=8192, k_len=8192, dim=256),
        # Cross-attention of a video model's block: every latent token over the text tokens.
        _case(name="text_cross_32k", q_heads=40, kv_heads=40, q_len=32760, k_len=512),
        # The masked benchmark (unequal lengths, outlier channels): a padded batch ...
        _case(name="key_padding", batch=2, q_heads=24, kv_heads=24, q_len=4096, k_len=4608, dim=64,
              mask="key_padding", inputs="outliers"),
        # ... an additive bias that the heads share ...
        _case(name="additive_bias", batch=2, q_heads=24, kv_heads=24, q_len=4096, k_len=4608,
              mask="bias", mask_dtype="fp32", inputs="outliers"),
        # ... and a boolean mask with rows that see no key, with the log-normalisers.
        _case(name="bool_mask_lse", batch=2, q_heads=24, kv_heads=24, q_len=4096, k_len=4608, dim=64,
              mask="bool", lse=True, inputs="outliers"),
        # Sparse path: the step of a sampling run that builds the pattern ...
        _case(name="construct_16k", path="construct", q_len=16384, k_len=16384, inputs="blocks"),
        # ... and one of those that reuse it (about half of the key tiles kept), inputs drifted.
        _case(name="reuse_32k", path="reuse", q_len=32768, k_len=32768, inputs="blocks"),
    ]


# Longest draws: the listed headline call is the most work, the listed video call the most bytes.
_MOST_OPS = 4 * 16 * 32768 * 32768 * 128
_MOST_BYTES = 1 << 29


def _length(rng, low, high):
    length = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    # sequence lengths are multiples of a tile about as often as they are not
    return max(low, length // 128 * 128) if rng.random() < 0.4 and length >= 128 else length


def draw(rng):
    """One more call: lengths over the whole range, ragged ones among them, every option."""
    case = _case()
    case["q_heads"], case["kv_heads"] = rng.choice([(16, 4), (16, 4), (32, 8), (24, 24), (8, 8), (40, 40), (16, 1), (12, 12)])
    case["batch"] = rng.choice([1, 1, 2, 4])
    case["dim"] = rng.choice([128, 128, 128, 64, 64, 256, 40, 80, 200])
    case["dtype"] = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    case["mode"] = rng.choice(["absmax", "absmax", "midpoint_affine"])
    case["nhd"] = rng.random() < 0.3
    kind = rng.choice(["self", "self", "self", "causal", "cross", "cross", "masked", "masked", "masked", "sparse",
                       "sparse", "split"])
    low, high = 64, 32768
    if kind == "self":
        case["q_len"] = case["k_len"] = _length(rng, low, high)
        case["lse"] = rng.random() < 0.2
    elif kind == "causal":
        case["causal"] = True
        case["q_len"] = case["k_len"] = _length(rng, low, high)
    elif kind == "cross":
        case["q_len"], case["k_len"] = _length(rng, low, high), _length(rng, low, 8192)
        case["lse"] = rng.random() < 0.2
    elif kind == "masked":
        case["mask"] = rng.choice(["key_padding", "key_padding", "key_bias", "bool", "bool", "bias", "bias",
                                   "documents", "window"])
        if case["mask"] in ("key_bias", "bias"):
            case["mask_dtype"] = rng.choice(["fp32", "bf16", "fp16"])
        case["inputs"] = rng.choice(["normal", "outliers"])
        case["q_len"], case["k_len"] = _length(rng, low, 8192), _length(rng, low, 8192)
        case["lse"] = rng.random() < 0.3
    elif kind == "sparse":
        case["path"] = rng.choice(["construct", "reuse"])
        case["inputs"] = "blocks"
        case["dim"] = rng.choice([128, 128, 64])
        case["q_len"] = case["k_len"] = _length(rng, 1024, high)
    else:
        case["path"] = "split"
        case["q_len"] = case["k_len"] = _length(rng, low, high)
    weight = {"none": 1, "key_padding": 1.5, "key_bias": 1.5}.get(case["mask"], 4)
    weight *= 2 if case["path"] == "construct" or case["dim"] == 200 else 1
    while True:
        ops = 4 * case["batch"] * case["q_heads"] * case["q_len"] * case["k_len"] * max(64, case["dim"])
        if ops * weight <= _MOST_OPS / 2 and work(case)["bytes"] <= _MOST_BYTES:
            return case
        case["q_len"] = max(64, int(case["q_len"] * 0.7))
        case["k_len"] = case["q_len"] if kind in ("self", "causal", "sparse", "split") else max(64, int(case["k_len"] * 0.7))


def _inputs(case, generator):
    """Q, K and V in float32 and the noise that drifts them between the steps of a sampling run."""
    b, hq, hkv, d = case["batch"], case["q_heads"], case["kv_heads"], case["dim"]

    def normal(heads, length):
        if case["nhd"]:
            return torch.randn(b, length, heads, d, generator=generator, device="cuda").transpose(1, 2)
        return torch.randn(b, heads, length, d, generator=generator, device="cuda")

    q, k, v = normal(hq, case["q_len"]), normal(hkv, case["k_len"]), normal(hkv, case["k_len"])
    if case["inputs"] == "outliers":  # one channel in a hundred twenty times as large
        hot = torch.randperm(d, generator=generator, device="cuda")[: max(1, d // 100)]
        for tensor in (q, k, v):
            tensor[..., hot] *= 20.0
    elif case["inputs"] == "blocks":  # 128-token blocks around one of two prototypes of norm 8
        prototypes = torch.randn(b, hkv, 2, d, generator=generator, device="cuda")
        prototypes *= 8.0 / prototypes.norm(dim=-1, keepdim=True)
        block = torch.arange(case["k_len"], device="cuda") // 128 % 2
        k += prototypes[:, :, block]
        q += prototypes.repeat_interleave(hq // hkv, 1)[:, :, block]
    return q, k, v


def _mask(case, generator):
    b, lq, lk, kind = case["batch"], case["q_len"], case["k_len"], case["mask"]
    if kind == "none":
        return None
    if kind == "key_padding":  # prompts of different lengths padded to one
        visible = torch.full((b,), lk, device="cuda")
        visible[b // 2:] = max(1, lk * 9 // 10)
        return (torch.arange(lk, device="cuda") < visible[:, None])[:, None, None]
    if kind == "key_bias":
        return torch.randn(b, 1, 1, lk, generator=generator, device="cuda").to(DTYPES[case["mask_dtype"]])
    if kind == "bias":
        return torch.randn(b, 1, lq, lk, generator=generator, device="cuda").to(DTYPES[case["mask_dtype"]])
    if kind == "bool":  # every key visible, but for a few rows that see none
        mask = torch.ones(b, 1, lq, lk, dtype=torch.bool, device="cuda")
        mask[0, :, :7] = False
        return mask
    rows = torch.arange(lq, device="cuda")[:, None]
    keys = torch.arange(lk, device="cuda")[None, :]
    if kind == "documents":  # eight packed documents
        return (rows * 8 // lq == keys * 8 // lk)[None, None].expand(b, 1, lq, lk).contiguous()
    return ((keys <= rows) & (keys > rows - 1024))[None, None].expand(b, 1, lq, lk).contiguous()  # window


def prepare(case, seed):
    case = {**DEFAULTS, **case}
    generator = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = DTYPES[case["dtype"]]
    q, k, v = _inputs(case, generator)
    state = {"case": case, "mask": _mask(case, generator), "pattern": None}
    if case["path"] == "reuse":  # the pattern of the run's first step, and inputs of a later one
        _, state["pattern"] = risa.construct_sparse_int8_attention(
            q.to(dtype), k.to(dtype), v.to(dtype), theta=0.99, v_quantization=case["mode"])
        for tensor in (q, k):
            tensor += 0.05 * torch.randn(tensor.shape, generator=generator, device="cuda")
    state["q"], state["k"], state["v"] = q.to(dtype), k.to(dtype), v.to(dtype)
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if case["path"] == "construct":
        out, pattern = risa.construct_sparse_int8_attention(q, k, v, theta=0.99, v_quantization=case["mode"])
        # (every run of one shape gives tensors of one shape: the lists are filled up with -1)
        free = pattern.rows * pattern.key_blocks - pattern.block_indices.numel()
        return out, pattern.row_offsets, torch.nn.functional.pad(pattern.block_indices, (0, free), value=-1)
    if case["path"] == "reuse":
        return risa.sparse_int8_attention(q, k, v, state["pattern"], v_quantization=case["mode"])
    if case["path"] == "split":
        packed = risa.prequantize_int8_attention(q, k, v, v_quantization=case["mode"])
        return risa.int8_attention_from_prequantized(packed, output_layout="nhd" if case["nhd"] else "hnd")
    return risa.int8_attention(q, k, v, attn_mask=state["mask"], v_quantization=case["mode"],
                               is_causal=case["causal"], return_lse=case["lse"])


def work(case):
    """Inputs and mask read once, outputs written once; the products of the visible scores."""
    case = {**DEFAULTS, **case}
    b, hq, hkv, lq, lk, d = (case[n] for n in ("batch", "q_heads", "kv_heads", "q_len", "k_len", "dim"))
    element = 4 if case["dtype"] == "fp32" else 2
    moved = element * d * b * (2 * hq * lq + 2 * hkv * lk)
    if case["lse"]:
        moved += 4 * b * hq * lq
    mask_element = 1 if case["mask_dtype"] == "bool" else 4 if case["mask_dtype"] == "fp32" else 2
    if case["mask"] in ("key_padding", "key_bias"):
        moved += mask_element * b * lk
    elif case["mask"] != "none":
        moved += mask_element * b * lq * lk
    scores = lq * lk
    if case["causal"]:
        seen = min(lq, lk)
        scores = seen * (seen + 1) // 2 + (lq - seen) * lk
    elif case["mask"] == "documents":
        scores //= 8
    elif case["mask"] == "window":
        scores = sum(max(0, min(row + 1, lk) - max(0, row - 1023)) for row in range(lq))
    elif case["mask"] == "key_padding":
        scores = (b // 2 * lk + (b - b // 2) * max(1, lk * 9 // 10)) * lq // b
    elif case["path"] == "reuse":  # half of the blocks share a query block's prototype
        scores //= 2
    return {"bytes": moved, "flops": 4 * b * hq * scores * d}


def tolerance(case):
    """Four times what the kernels differ from the NumPy oracle by (the same arithmetic with exact
    exponentials and sums in another order): 4.8e-5 at most over 28 draws, single values by one
    bfloat16 step.  Pattern rows and tile lists are whole numbers and stay the same."""
    return {"rel": 2e-4, "max": 0.03}
