"""The work that a user of this package has it do, as cases that can be timed and compared.

Five kinds, each through the public entry points a user's program calls:

  attention  ``decode_attention``: one query token per sequence against a KV cache, a global or a sliding-window layer
  experts    ``decode_gemm`` twice: a MoE layer's up projection with fused SwiGLU, then its down projection
  dense      ``quant.dot`` (or ``decode_gemm`` with SwiGLU for an up projection): one dense projection of a layer
  head       ``quant.dot`` to float32 logits over the padded vocabulary, then the greedy ``sample_token``
  step       a whole decode step: ``model_apply`` and ``sample_token`` call by call, or a ``GraphedDecoder`` replay

Widths, head counts, expert counts and windows are those of ``lyra_amd.model.MODEL_VARIANTS``; batches and contexts are the
ones a decode loop meets, from one sequence to 128 and from a short prompt to 4096 tokens, odd sizes among them.
"""
from __future__ import annotations

import math
import os
from dataclasses import replace

os.environ.setdefault("LYRA_LOG_KERNELS", "0")  # a serving process switches the per-shape log lines off

import numpy as np  # noqa: E402
import torch  # noqa: E402

from lyra_amd.generate import GraphedDecoder, sample_token  # noqa: E402
from lyra_amd.kernels.decode_attention import decode_attention  # noqa: E402
from lyra_amd.kernels.decode_gemm import decode_gemm  # noqa: E402
from lyra_amd.model import (  # noqa: E402
    MODEL_VARIANTS,
    LayerCache,
    ModelCache,
    apply_inference_overrides,
    init_weights,
    interleaved_moe,
    model_apply,
)
from lyra_amd.nn.quant import QArray, dot, quantize  # noqa: E402

FP8 = torch.float8_e4m3fn
DEVICE = "cuda:0"

# query heads, kv heads, head width of the attention layers of the variants; whether they have an output gate
HEADS = {
    "dev": (2, 1, 64, False),
    "lyra-small": (16, 4, 128, True),
    "lyra-medium": (32, 8, 128, True),
    "gpt-oss-20b": (64, 8, 64, False),
}


def listed():
    return [
        # one user at a prompt, early in the conversation: the smallest call there is
        dict(name="attention-b1-bf16", kind="attention", heads="lyra-small", batch=1, length=512, cache="bf16", window=0, ragged=False),
        # a full serving batch at full context on a global layer (every second layer of a model)
        dict(name="attention-b64-fp8", kind="attention", heads="lyra-small", batch=64, length=4096, cache="fp8", window=0, ragged=False),
        # continuous batching: every sequence at its own position, cache length not a multiple of anything
        dict(name="attention-b48-ragged", kind="attention", heads="gpt-oss-20b", batch=48, length=3001, cache="fp8", window=0, ragged=True),
        # a fused q/k/v projection for a handful of sequences, weights as trained
        dict(name="dense-qkv-m5-bf16", kind="dense", variant="lyra-small", proj="qkv", rows=5, weights="bf16"),
        # a MoE layer for a few sequences, weights as trained
        dict(name="experts-small-t7-bf16", kind="experts", variant="lyra-small", tokens=7, weights="bf16"),
        # a MoE layer of the middle variant at a serving batch, scale blocks as the reference's --fp8 quantises
        dict(name="experts-medium-t64-fp8", kind="experts", variant="lyra-medium", tokens=64, weights="fp8-block"),
        # widths that are not a multiple of 128, biases, no shared expert
        dict(name="experts-gptoss-t33-fp8", kind="experts", variant="gpt-oss-20b", tokens=33, weights="fp8-channel"),
        # the LM head and the choice of the next token for a batch of more than one 64-row block
        dict(name="head-m96-bf16", kind="head", variant="lyra-small", rows=96),
        # the interactive loop: one sequence, every operator called from Python, nothing quantised
        dict(name="step-small-b1-bf16", kind="step", variant="lyra-small", batch=1, context=1000, layout="bf16", graph=False),
        # a few sequences in the layout the reference's --fp8 sets, captured in a graph
        dict(name="step-small-b8-fp8", kind="step", variant="lyra-small", batch=8, context=2048, layout="serve", graph=True),
        # the benchmark's headline step
        dict(name="step-small-b64-fp8", kind="step", variant="lyra-small", batch=64, context=4096, layout="fp8", graph=True),
        # a large batch of the middle variant (exclusive self attention; eight of its layers, so that three states fit)
        dict(name="step-medium-b128-fp8", kind="step", variant="lyra-medium", batch=128, context=1500, layout="fp8", graph=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_MOST_BYTES = None


def draw(rng):
    global _MOST_BYTES
    if _MOST_BYTES is None:
        _MOST_BYTES = max(work(c)["bytes"] for c in listed())
    while True:
        kind = rng.choice(["attention", "attention", "experts", "experts", "dense", "head", "step", "step"])
        if kind == "attention":
            case = dict(kind=kind, heads=rng.choice(["lyra-small", "lyra-medium", "gpt-oss-20b"]), batch=_log_int(rng, 1, 128),
                        length=_log_int(rng, 64, 4096), cache=rng.choice(["bf16", "fp8", "fp8"]), window=rng.choice([0, 0, 128]),
                        ragged=rng.choice([False, True]))
        elif kind == "experts":
            case = dict(kind=kind, variant=rng.choice(["lyra-small", "lyra-medium", "lyra-max", "gpt-oss-20b"]),
                        tokens=_log_int(rng, 1, 128), weights=rng.choice(["bf16", "fp8-block", "fp8-channel"]))
            if case["variant"] == "gpt-oss-20b" and case["weights"] == "fp8-block":
                case["weights"] = "fp8-channel"  # (2880 has no 256-wide blocks)
            if case["variant"] == "lyra-max" and case["weights"] == "bf16":
                case["weights"] = "fp8-block"  # (served quantised only)
        elif kind == "dense":
            case = dict(kind=kind, variant=rng.choice(["lyra-small", "lyra-medium", "gpt-oss-20b"]), proj=rng.choice(["qkv", "out", "up", "down"]),
                        rows=_log_int(rng, 1, 256), weights=rng.choice(["bf16", "fp8-block", "fp8-channel"]))
            if case["variant"] == "gpt-oss-20b":
                case["proj"] = rng.choice(["qkv", "out"])  # (every MLP of it is a MoE layer)
                if case["weights"] == "fp8-block":
                    case["weights"] = "fp8-channel"
        elif kind == "head":
            case = dict(kind=kind, variant=rng.choice(["lyra-small", "lyra-medium", "gpt-oss-20b"]), rows=_log_int(rng, 1, 128))
        else:
            variant = rng.choice(["dev", "lyra-small", "lyra-small", "lyra-small"])
            layout = "bf16" if variant == "dev" else rng.choice(["bf16", "serve", "fp8"])
            case = dict(kind=kind, variant=variant, batch=_log_int(rng, 1, 32 if layout == "bf16" else 128),
                        context=_log_int(rng, 16, 256) if variant == "dev" else _log_int(rng, 128, 4096), layout=layout,
                        graph=rng.choice([False, True]))
        if work(case)["bytes"] <= _MOST_BYTES:
            return case


# ---- shapes ------------------------------------------------------------------------------------------------------
def _model_config(case):
    cfg = MODEL_VARIANTS[case["variant"]]
    if case["variant"] == "lyra-medium":
        cfg = replace(cfg, n_layers=8, mlp_map=interleaved_moe(8, first=4, every=4))
    if case["layout"] == "serve":  # what the reference's --fp8 sets
        cfg = apply_inference_overrides(cfg, fp8=True)
    elif case["layout"] == "fp8":  # the benchmark's layout: attention projections too, one scale per output channel
        cfg = apply_inference_overrides(cfg, fp8=True, fp8_attn=True, per_channel=True)
    return replace(cfg, sample_temperature=0.0)


def _dense_shape(case):
    """(rows of the weight, columns, SwiGLU behind it) of a dense projection."""
    cfg = MODEL_VARIANTS[case["variant"]]
    heads = cfg.n_attn_heads * cfg.head_dim
    return {
        "qkv": (cfg.n_embd, heads + 2 * cfg.n_kv_heads * cfg.head_dim, False),
        "out": (heads, cfg.n_embd, False),
        "up": (cfg.n_embd, 2 * cfg.dense_hidden, True),
        "down": (cfg.dense_hidden, cfg.n_embd, False),
    }[case["proj"]]


def _scale_block(weights, k, n):
    return (k, 1) if weights == "fp8-channel" else (math.gcd(k, 256), math.gcd(n, 256))


def _weight_bytes(weights, k, n):
    if weights == "bf16":
        return 2 * k * n
    bk, bn = _scale_block(weights, k, n)
    return k * n + 4 * (k // bk) * (n // bn)


def _group_sizes(cfg, tokens, rng):
    """Rows per expert when every token picks its routed experts with p_i ~ i^-1.1 (trained routers are skewed) and every
    shared one."""
    p = 1.0 / np.arange(1, cfg.n_routed_experts + 1) ** 1.1
    # the k largest of log p + Gumbel noise are k distinct experts drawn in proportion to p
    keys = np.log(p) + rng.gumbel(size=(tokens, cfg.n_routed_experts))
    ids = np.argsort(-keys, axis=1)[:, : cfg.n_active_routed_experts]
    sizes = np.bincount(ids.reshape(-1), minlength=cfg.n_experts).astype(np.int32)
    sizes[cfg.n_routed_experts :] = tokens
    return sizes


def _visible(case, position):
    return min(position + 1, case["window"]) if case["window"] else position + 1


# ---- states ------------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _weights(g, kind, groups, k, n):
    w = torch.empty(groups, k, n, device=DEVICE, dtype=torch.bfloat16).normal_(0.0, 0.02, generator=g)
    return w if kind == "bf16" else quantize(w, FP8, _scale_block(kind, k, n))


def _cache_rows(g, shape, fp8):
    """A cache with a history: bf16 rows ~ N(0, 1), or FP8 codes with the scales of such rows."""
    if not fp8:
        return torch.empty(shape, device=DEVICE, dtype=torch.bfloat16).normal_(generator=g)
    codes = torch.empty(shape, device=DEVICE, dtype=torch.uint8)
    for row in codes:  # (a layer or a sequence at a time: no large temporaries)
        row.copy_((torch.empty(row.shape, device=DEVICE, dtype=torch.bfloat16).normal_(0.0, 140.0, generator=g)).clamp_(-448, 448).to(FP8).view(torch.uint8))
    scale = torch.rand(*shape[:-1], 1, device=DEVICE, generator=g) * 0.004 + 0.006
    return QArray(codes.view(FP8), scale, (1, shape[-1]))


def _prepare_attention(case, seed):
    g = _generator(seed)
    n, k, h, gated = HEADS[case["heads"]]
    b, s = case["batch"], case["length"]
    shape = (b, k, s, h)
    if case["ragged"]:
        position = torch.randint(min(s - 1, s // 16), s, (b,), device=DEVICE, generator=g).to(torch.int32)
    else:
        position = torch.tensor(s - 1, dtype=torch.int32, device=DEVICE)
    return dict(
        q=torch.empty(b, n, 1, h, device=DEVICE, dtype=torch.bfloat16).normal_(generator=g),
        k=_cache_rows(g, shape, case["cache"] == "fp8"), v=_cache_rows(g, shape, case["cache"] == "fp8"),
        sinks=torch.empty(n, device=DEVICE).normal_(generator=g), position=position, window=case["window"], scale=h**-0.5,
        gate=(2 * torch.sigmoid(torch.empty(b, n, device=DEVICE).normal_(generator=g))).to(torch.bfloat16) if gated else None,
    )


def _prepare_experts(case, seed):
    g = _generator(seed)
    cfg = MODEL_VARIANTS[case["variant"]]
    sizes = _group_sizes(cfg, case["tokens"], np.random.default_rng(seed))
    e, c, hd = cfg.n_experts, cfg.n_embd, cfg.expert_hidden
    bias = lambda n: torch.empty(e, n, device=DEVICE).normal_(0.0, 0.5, generator=g) if cfg.use_mlp_bias else None  # noqa: E731
    return dict(
        rows=torch.empty(int(sizes.sum()), c, device=DEVICE, dtype=torch.bfloat16).normal_(generator=g),
        sizes=torch.from_numpy(sizes).to(DEVICE), up=_weights(g, case["weights"], e, c, 2 * hd), down=_weights(g, case["weights"], e, hd, c),
        up_bias=bias(2 * hd), down_bias=bias(c), quant=None if case["weights"] == "bf16" else FP8,
    )


def _prepare_dense(case, seed):
    g = _generator(seed)
    k, n, swiglu = _dense_shape(case)
    w = _weights(g, case["weights"], 1, k, n)
    if not swiglu:
        w = QArray(w.qval[0], w.scale[0], w.block) if isinstance(w, QArray) else w[0]
    return dict(rows=torch.empty(case["rows"], k, device=DEVICE, dtype=torch.bfloat16).normal_(generator=g), w=w, swiglu=swiglu,
                sizes=torch.full((1,), case["rows"], dtype=torch.int32, device=DEVICE), quant=None if case["weights"] == "bf16" else FP8)


def _prepare_head(case, seed):
    g = _generator(seed)
    cfg = MODEL_VARIANTS[case["variant"]]
    return dict(rows=torch.empty(case["rows"], cfg.n_embd, device=DEVICE, dtype=torch.bfloat16).normal_(generator=g),
                w=_weights(g, "bf16", 1, cfg.n_embd, cfg.padded_vocab_size)[0], cfg=replace(cfg, sample_temperature=0.0))


def _prepare_step(case, seed):
    cfg = _model_config(case)
    b, s = case["batch"], case["context"]
    g = _generator(seed + 1)
    model = init_weights(cfg, DEVICE, seed)
    # A trained model's embeddings are not small beside what its layers add to them, and its routers are decided: rows of
    # unit size instead of init_weights' 0.02, router biases of a trained model's spread.  (With the fresh values the bf16
    # rounding of the residual stream grows to 2-4 % of the logits by the last layer, and tokens change experts on it.)
    model.emb.mul_(1.0 / cfg.w_std)
    for layer in model.layers:
        if getattr(layer.mlp, "router_bias", None) is not None:
            layer.mlp.router_bias.normal_(generator=g)
    shape = (cfg.n_layers, b, cfg.n_kv_heads, s, cfg.head_dim)
    stacks = [_cache_rows(g, shape, cfg.quantize_cache) for _ in range(2)]

    def layer_rows(stack, i):
        return QArray(stack.qval[i], stack.scale[i], stack.block) if isinstance(stack, QArray) else stack[i]

    cache = ModelCache([LayerCache(layer_rows(stacks[0], i), layer_rows(stacks[1], i)) for i in range(cfg.n_layers)],
                       torch.tensor(s - 1, dtype=torch.int32, device=DEVICE))
    tokens = torch.randint(0, cfg.vocab_size, (b,), device=DEVICE, generator=g).to(torch.int32)
    # the position stays where it is, so that every pass decodes at the same context
    decoder = GraphedDecoder(model, cache, cfg, b, advance=False) if case["graph"] else None
    return dict(cfg=cfg, model=model, cache=cache, stacks=stacks, tokens=tokens, decoder=decoder)


def prepare(case, seed):
    make = {"attention": _prepare_attention, "experts": _prepare_experts, "dense": _prepare_dense, "head": _prepare_head, "step": _prepare_step}
    return dict(make[case["kind"]](case, seed), kind=case["kind"])


# ---- one pass ----------------------------------------------------------------------------------------------------
def run(s):
    if s["kind"] == "attention":
        return decode_attention(s["q"], s["k"], s["v"], s["sinks"], s["scale"], s["window"], s["position"], gate=s["gate"])
    if s["kind"] == "experts":
        hidden = decode_gemm(s["rows"], s["up"], s["sizes"], bias=s["up_bias"], fused_swiglu=True, quant_dtype=s["quant"])
        return hidden, decode_gemm(hidden, s["down"], s["sizes"], bias=s["down_bias"], quant_dtype=s["quant"])
    if s["kind"] == "dense":
        if s["swiglu"]:
            return decode_gemm(s["rows"], s["w"], s["sizes"], fused_swiglu=True, quant_dtype=s["quant"])
        return dot(s["rows"], s["w"])
    if s["kind"] == "head":
        logits = dot(s["rows"], s["w"], preferred_element_type=torch.float32)
        return logits, sample_token(logits, s["cfg"])
    if s["decoder"] is not None:
        s["decoder"].tokens.copy_(s["tokens"])
        s["decoder"].step()
        logits = s["decoder"].logits
    else:
        logits, _ = model_apply(s["tokens"], s["model"], s["cache"], s["cfg"], advance=False)
        sample_token(logits, s["cfg"])
    # (the drawn tokens follow from the logits; the caches hold the new rows)
    return dict(logits=logits,
                caches=[(t.qval.view(torch.uint8), t.scale) if isinstance(t, QArray) else t for t in s["stacks"]])


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _attention_work(batch, n, k, h, keys, fp8):
    """`keys`: visible keys of all sequences together."""
    per_key = h * (1 if fp8 else 2) + (4 if fp8 else 0)
    return 2 * k * keys * per_key + 4 * batch * n * h, 4 * n * h * keys


def _experts_work(cfg, tokens, weights):
    sizes = _group_sizes(cfg, tokens, np.random.default_rng(0))
    touched, rows = int((sizes > 0).sum()), int(sizes.sum())
    c, hd = cfg.n_embd, cfg.expert_hidden
    nbytes = touched * (_weight_bytes(weights, c, 2 * hd) + _weight_bytes(weights, hd, c)) + 2 * rows * (2 * c + 2 * hd)
    return nbytes, 2 * rows * (c * 2 * hd + hd * c)


def _step_work(case):
    cfg = _model_config(case)
    b, s, c = case["batch"], case["context"], cfg.n_embd
    mlp = {"bf16": "bf16", "serve": "fp8-block", "fp8": "fp8-channel"}[case["layout"]]
    attn = "fp8-channel" if case["layout"] == "fp8" else "bf16"
    heads = cfg.n_attn_heads * cfg.head_dim
    width = heads + 2 * cfg.n_kv_heads * cfg.head_dim
    nbytes, flops = 2 * c * cfg.padded_vocab_size + 4 * b * cfg.padded_vocab_size, 2 * b * c * cfg.padded_vocab_size
    for i in range(cfg.n_layers):
        keys = min(s, cfg.sliding_window) if i % 2 == 0 and cfg.sliding_window else s
        a_bytes, a_flops = _attention_work(b, cfg.n_attn_heads, cfg.n_kv_heads, cfg.head_dim, b * keys, cfg.quantize_cache)
        nbytes += a_bytes + _weight_bytes(attn, c, width) + _weight_bytes(attn, heads, c)
        flops += a_flops + 2 * b * c * (width + heads)
        if cfg.mlp_map[i] == "moe":
            m_bytes, m_flops = _experts_work(cfg, b, mlp)
        else:
            hd = cfg.dense_hidden
            m_bytes, m_flops = _weight_bytes(mlp, c, 2 * hd) + _weight_bytes(mlp, hd, c), 6 * b * c * hd
        nbytes += m_bytes
        flops += m_flops
    return nbytes, flops


def work(case):
    if case["kind"] == "attention":
        n, k, h, _ = HEADS[case["heads"]]
        b, s = case["batch"], case["length"]
        # (ragged: positions uniform over the upper 15/16 of the cache)
        mean = _visible(case, (min(s - 1, s // 16) + s - 1) / 2) if case["ragged"] else _visible(case, s - 1)
        nbytes, flops = _attention_work(b, n, k, h, b * mean, case["cache"] == "fp8")
    elif case["kind"] == "experts":
        nbytes, flops = _experts_work(MODEL_VARIANTS[case["variant"]], case["tokens"], case["weights"])
    elif case["kind"] == "dense":
        k, n, swiglu = _dense_shape(case)
        m = case["rows"]
        nbytes, flops = _weight_bytes(case["weights"], k, n) + 2 * m * (k + (n // 2 if swiglu else n)), 2 * m * k * n
    elif case["kind"] == "head":
        cfg = MODEL_VARIANTS[case["variant"]]
        m, v = case["rows"], cfg.padded_vocab_size
        nbytes, flops = 2 * cfg.n_embd * (v + m) + 4 * m * v, 2 * m * cfg.n_embd * v
    else:
        nbytes, flops = _step_work(case)
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    """About four times what was seen against a float64 restatement on the same inputs (attention 0.0029, matmuls 0.0027 and
    head 2.7e-7 in the 2-norm), and for whole steps against the plain-operator driver, which rounds at other places: 0.0058,
    up to 0.014 where a token near a tie changes its expert."""
    if case["kind"] == "head":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}  # (two logits of a row may tie to the last bits)
    if case["kind"] == "attention":
        return {"rel": 1e-2, "max": 0.06}
    if case["kind"] == "step":
        return {"rel": 2.4e-2, "max": 0.9, "differ": min(0.01, 1.0 / case["context"])}  # (codes of the one new row per cache)
    return {"rel": 1e-2, "max": 0.08}
