"""What a user of this framework has it do, as cases to measure: the products, the Gemma2 MLP and output head, the attention of a
prompt and of a generation step, the attention scores' softmax and the Zamba2 mixer's convolution and norm, each through
`anygpu_amd.ops` on tensors that already are on the device.

Shapes are those of the repository's own benchmark and tests (layer weights, head counts, head dimensions), row counts and
sequence lengths run over the range a serving program meets: one sequence generating up to a prompt of a few thousand tokens.
Values follow the same places: activations N(0, 1), weights N(0, 1 / K), attention scores N(0, 16).
"""
from __future__ import annotations

import math

import torch

from anygpu_amd import capi, ops

DTYPES = {"f16": torch.float16, "f32": torch.float32}

# (n, k) of a layer's projections, (hidden, intermediate) of an MLP, (vocabulary, hidden) of an output head
LAYER_WEIGHTS = [(9216, 2304), (2304, 9216), (2048, 2304), (1024, 2304), (4096, 2304), (2304, 2048), (2048, 2048), (8192, 2048),
                 (2048, 8192), (4096, 4096), (14336, 4096), (4096, 14336), (6144, 4096), (18944, 3584)]
MLPS = [(2304, 9216), (2048, 8192), (3584, 14336), (4096, 14336)]
HEADS = [(256000, 2304), (128256, 4096), (131072, 2048)]
# (query heads, key / value heads, head dimension)
ATTENTION = [(8, 4, 256), (8, 1, 256), (16, 16, 128), (32, 8, 128), (64, 8, 128), (32, 32, 64), (16, 16, 64)]


def listed() -> list[dict]:
    return [
        # the smallest product: a float32 [256, 512] x [512, 1024], both operands as they lie in a row-major program
        {"name": "product f32 small", "kind": "product", "dtype": "f32", "m": 256, "n": 1024, "k": 512, "layout": "kn", "bias": False},
        # the large square half product, right operand stored [N, K]
        {"name": "product f16 4096", "kind": "product", "dtype": "f16", "m": 4096, "n": 4096, "k": 4096, "layout": "nk", "bias": False},
        # the Gemma2 MLP for the next token of eight sequences, weights as checkpoints hold them ([out, in])
        {"name": "mlp generation", "kind": "mlp", "dtype": "f16", "rows": 8, "hidden": 2304, "inter": 9216, "layout": "nk"},
        # the same for a prompt, weights in the layout of tensor_linear ([in, out])
        {"name": "mlp prompt", "kind": "mlp", "dtype": "f16", "rows": 1500, "hidden": 2304, "inter": 9216, "layout": "kn"},
        # the Gemma2 output head with its softcap, next token of eight sequences
        {"name": "output head generation", "kind": "head", "dtype": "f16", "rows": 8, "vocab": 256000, "hidden": 2304, "softcap": 30.0},
        # attention scores of a Gemma2 local layer over 8192 positions
        {"name": "scores softmax", "kind": "softmax", "dtype": "f16", "heads": 8, "q": 8192, "k": 8192, "softcap": 50.0, "window": 4096},
        # a Zamba2 mixer over four prompts: causal convolution + SiLU in front of the scan, gated norm behind it
        {"name": "mixer prompt", "kind": "mixer", "dtype": "f16", "batch": 4, "seq": 4096, "inner": 4096, "state": 64},
        # the same for one generated token of four sequences: the shortest call of the framework
        {"name": "mixer generation", "kind": "mixer step", "dtype": "f16", "batch": 4, "inner": 4096, "state": 64},
        # attention of a Gemma2 local layer over a long prompt
        {"name": "attention gemma2 prompt", "kind": "attention", "dtype": "f16", "batch": 1, "heads": 8, "kv_heads": 4, "dim": 256,
         "n_q": 8192, "n_k": 8192, "softcap": 50.0, "window": 4096, "causal": True},
        # attention over a prompt of ordinary length, grouped heads of dimension 128
        {"name": "attention prompt", "kind": "attention", "dtype": "f16", "batch": 1, "heads": 32, "kv_heads": 8, "dim": 128,
         "n_q": 3000, "n_k": 3000, "softcap": 0.0, "window": 0, "causal": True},
        # attention of one generated token, four sequences with five thousand cached positions each
        {"name": "attention generation", "kind": "attention", "dtype": "f16", "batch": 4, "heads": 32, "kv_heads": 8, "dim": 128,
         "n_q": 1, "n_k": 5001, "softcap": 0.0, "window": 0, "causal": True},
        # attention in float32 with the mask handed over as a tensor
        {"name": "attention mask f32", "kind": "masked", "dtype": "f32", "heads": 8, "dim": 256, "n_q": 3001, "n_k": 3001, "mask": "causal"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_any(rng) -> dict:
    kind = rng.choice(("product", "product", "mlp", "head", "softmax", "mixer", "mixer step", "attention", "attention", "attention", "masked"))
    half = "f16" if rng.random() < 0.7 else "f32"
    layout = rng.choice(("nk", "kn"))
    if kind == "product":
        if rng.random() < 0.3:      # any sizes at all
            m, n, k = (_log_int(rng, 128, 4096) for _ in range(3))
        else:                       # a layer's projection of any number of tokens
            m = _log_int(rng, 1, 4096)
            n, k = rng.choice(LAYER_WEIGHTS)
        return {"kind": kind, "dtype": half, "m": m, "n": n, "k": k, "layout": layout, "bias": rng.random() < 0.25}
    if kind == "mlp":
        hidden, inter = rng.choice(MLPS)
        return {"kind": kind, "dtype": half, "rows": _log_int(rng, 1, 4096), "hidden": hidden, "inter": inter, "layout": layout}
    if kind == "head":
        vocab, hidden = rng.choice(HEADS)
        return {"kind": kind, "dtype": half, "rows": _log_int(rng, 1, 64), "vocab": vocab, "hidden": hidden, "softcap": 30.0}
    if kind == "softmax":
        heads, q = rng.choice((1, 8, 16, 32)), _log_int(rng, 64, 8192)
        capped = rng.random() < 0.5
        return {"kind": kind, "dtype": half, "heads": heads, "q": q, "k": q if rng.random() < 0.7 else _log_int(rng, q, 16384),
                "softcap": 50.0 if capped else 0.0, "window": rng.choice((0, 4096)) if capped else 0}
    if kind in ("mixer", "mixer step"):
        inner = rng.choice((2048, 4096, 8192))
        if kind == "mixer step":
            return {"kind": kind, "dtype": half, "batch": _log_int(rng, 1, 256), "inner": inner, "state": 64}
        return {"kind": kind, "dtype": half, "batch": rng.choice((1, 2, 4)), "seq": _log_int(rng, 16, 8192), "inner": inner, "state": 64}
    heads, kv_heads, dim = rng.choice(ATTENTION)
    if kind == "masked":
        n_q = _log_int(rng, 16, 4096)
        return {"kind": kind, "dtype": "f32" if rng.random() < 0.6 else "f16", "heads": heads, "dim": dim, "n_q": n_q,
                "n_k": n_q if rng.random() < 0.7 else _log_int(rng, n_q, 8192), "mask": rng.choice(("causal", "causal", "window", "bias"))}
    capped = dim == 256 and rng.random() < 0.7
    case = {"kind": kind, "dtype": half, "batch": rng.choice((1, 1, 2, 4)), "heads": heads, "kv_heads": kv_heads, "dim": dim, "n_q": 1, "n_k": 1,
            "softcap": 50.0 if capped else 0.0, "window": rng.choice((0, 4096)) if capped else 0, "causal": True}
    shape = rng.random()
    if shape < 0.5:                 # a prompt; sometimes without the causal rule, as an encoder has it
        case["n_q"] = case["n_k"] = _log_int(rng, 64, 8192)
        case["causal"] = rng.random() < 0.85 or case["window"] > 0
    elif shape < 0.65:              # a chunk of a prompt against what is cached
        case["n_q"] = _log_int(rng, 64, 1024)
        case["n_k"] = _log_int(rng, 2 * case["n_q"], 32768)
    else:                           # one generated token, or a few that are checked together
        case["n_q"] = rng.choice((1, 1, 1, 2, 4))
        case["n_k"] = _log_int(rng, 256, 32768)
    return case


def _cost_us(case: dict) -> float:
    """Rough time of a pass, to keep drawn cases below the largest listed ones."""
    w = work(case)
    rate = 5e14 if case["dtype"] == "f16" else 1e14
    return 1e6 * (w["bytes"] / 5e12 + w["flops"] / rate)


def draw(rng) -> dict:
    while True:
        case = _draw_any(rng)
        if _cost_us(case) <= 450.0:
            return case


def _visible_pairs(n_q: int, n_k: int, causal: bool, window: int) -> int:
    """(query, key) pairs that the index rules leave, query i standing at key i + n_k - n_q."""
    if not causal:
        return n_q * n_k
    total = 0
    for i in range(n_q):
        total += min(i + n_k - n_q + 1, window) if window else i + n_k - n_q + 1
    return total


def work(case: dict) -> dict:
    es = 2 if case["dtype"] == "f16" else 4
    kind = case["kind"]
    if kind == "product":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (m * k + n * k + m * n + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    if kind == "mlp":
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        return {"bytes": es * (3 * hidden * inter + 2 * rows * hidden), "flops": 6 * rows * hidden * inter}
    if kind == "head":
        rows, vocab, hidden = case["rows"], case["vocab"], case["hidden"]
        return {"bytes": es * (vocab * hidden + rows * (vocab + hidden)), "flops": 2 * rows * vocab * hidden}
    if kind == "softmax":
        visible = case["heads"] * _visible_pairs(case["q"], case["k"], True, case["window"])
        return {"bytes": es * (visible + case["heads"] * case["q"] * case["k"]), "flops": 8 * visible}
    if kind in ("mixer", "mixer step"):
        dims, inner = case["inner"] + 2 * case["state"], case["inner"]
        if kind == "mixer":
            tokens = case["batch"] * case["seq"]
            return {"bytes": es * (tokens * (2 * dims + 3 * inner) + 5 * dims + inner), "flops": tokens * (12 * dims + 8 * inner)}
        tokens = case["batch"]
        return {"bytes": es * (tokens * (8 * dims + 3 * inner) + 5 * dims + inner), "flops": tokens * (12 * dims + 8 * inner)}
    n_q, n_k, d = case["n_q"], case["n_k"], case["dim"]
    if kind == "masked":
        pairs = n_q * n_k if case["mask"] == "bias" else _visible_pairs(n_q, n_k, True, 1024 if case["mask"] == "window" else 0)
        return {"bytes": es * (2 * case["heads"] * d * (n_q + n_k) + n_q * n_k), "flops": 4 * d * case["heads"] * pairs}
    pairs = _visible_pairs(n_q, n_k, case["causal"], case["window"])
    keys = min(n_k, case["window"] + n_q - 1) if case["window"] else n_k
    return {"bytes": es * 2 * case["batch"] * d * (case["heads"] * n_q + case["kv_heads"] * keys), "flops": 4 * d * case["batch"] * case["heads"] * pairs}


def prepare(case: dict, seed: int) -> dict:
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(*shape, std=1.0):
        t = torch.empty(shape, dtype=dtype, device="cuda")
        return t.normal_(0.0, std, generator=gen)

    def weight(n, k, layout="nk"):
        return normal(*((n, k) if layout == "nk" else (k, n)), std=k ** -0.5)

    kind = case["kind"]
    state = {"case": case, "layout": capi.B_COL_MAJOR if case.get("layout") == "nk" else capi.B_ROW_MAJOR}
    if kind == "product":
        state.update(x=normal(case["m"], case["k"]), w=weight(case["n"], case["k"], case["layout"]))
        if case["bias"]:
            state.update(b=normal(case["n"], std=0.1))
    elif kind == "mlp":
        hidden, inter, layout = case["hidden"], case["inter"], case["layout"]
        state.update(x=normal(case["rows"], hidden), gate=weight(inter, hidden, layout), up=weight(inter, hidden, layout),
                     down=weight(hidden, inter, layout))
    elif kind == "head":
        state.update(x=normal(1, case["rows"], case["hidden"]), w=weight(case["vocab"], case["hidden"]))
    elif kind == "softmax":
        state.update(x=normal(case["heads"] * case["q"], case["k"], std=16.0))
    elif kind in ("mixer", "mixer step"):
        inner, dims, batch = case["inner"], case["inner"] + 2 * case["state"], case["batch"]
        state.update(w=normal(dims, 4, std=0.5), b=normal(dims, std=0.1), norm=1.0 + normal(inner, std=0.1))
        if kind == "mixer":
            state.update(x=normal(batch, dims, case["seq"]), scan=normal(batch, case["seq"], inner), gate=normal(batch, case["seq"], inner))
        else:
            state.update(x=normal(batch, dims), past=normal(batch, dims, 3), scan=normal(batch, inner), gate=normal(batch, inner))
    elif kind == "masked":
        heads, d, n_q, n_k = case["heads"], case["dim"], case["n_q"], case["n_k"]
        state.update(q=normal(1, heads, n_q, d), k=normal(1, heads, n_k, d), v=normal(1, heads, n_k, d))
        if case["mask"] == "bias":
            mask = normal(n_q, n_k)
        else:
            at = torch.arange(n_q, device="cuda").unsqueeze(1) + (n_k - n_q)
            key = torch.arange(n_k, device="cuda").unsqueeze(0)
            hidden = key > at
            if case["mask"] == "window":
                hidden |= key <= at - 1024
            mask = torch.zeros(n_q, n_k, dtype=dtype, device="cuda").masked_fill_(hidden, -math.inf)
        state.update(mask=mask.reshape(1, 1, n_q, n_k))
    else:
        batch, d = case["batch"], case["dim"]
        state.update(q=normal(batch, case["heads"], case["n_q"], d), k=normal(batch, case["kv_heads"], case["n_k"], d),
                     v=normal(batch, case["kv_heads"], case["n_k"], d))
    return state


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "product":
        if case["bias"]:
            return ops.tensor_gemm(state["x"], state["w"], state["b"], b_layout=state["layout"])
        return ops.tensor_mm(state["x"], state["w"], b_layout=state["layout"])
    if kind == "mlp":
        up = ops.mlp_gemma2_fused_upproj(state["x"], state["gate"], state["up"], b_layout=state["layout"])
        return ops.tensor_mm(up, state["down"], b_layout=state["layout"])
    if kind == "head":
        return ops.tensor_gemma_linear_softcap(state["x"], state["w"], case["softcap"])
    if kind == "softmax":
        return ops.tensor_softmax(state["x"], alpha=1.0 / 16.0, softcap=case["softcap"], causal=True, window=case["window"],
                                  q_len=case["q"], diag=case["k"] - case["q"])
    if kind == "mixer":
        return (ops.tensor_causal_conv1d(state["x"], state["w"], state["b"]),
                ops.tensor_zamba_gated_rmsnorm(state["scan"], state["gate"], state["norm"], case["inner"], 1e-5))
    if kind == "mixer step":
        y = ops.tensor_causal_conv1d_update(state["x"], state["past"], state["w"], state["b"])
        return y, state["past"], ops.tensor_zamba_gated_rmsnorm(state["scan"], state["gate"], state["norm"], case["inner"], 1e-5)
    alpha = case["dim"] ** -0.5
    if kind == "masked":
        return ops.sdp_attention_masked_scaled_fwd(state["q"], state["k"], state["v"], state["mask"], alpha)
    return ops.sdp_attention_fwd(state["q"], state["k"], state["v"], alpha, softcap=case["softcap"], causal=case["causal"], window=case["window"])


def tolerance(case: dict):
    """About four times the error that these paths show against the same arithmetic in 64 bits: half results up to 2.9e-4 (2-norm) and
    1.8e-3 (largest), float32 results up to 1.1e-6 and 8e-6."""
    return {"rel": 1.2e-3, "max": 7e-3} if case["dtype"] == "f16" else {"rel": 4.5e-6, "max": 3.5e-5}
