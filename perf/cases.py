"""What this framework is used for, as cases that can be timed: prefill, training and decode of fused attention.

Every case builds the engine a user's program builds once per layer type (``AttentionEngine``, traced from the
script-level ``score_mod`` / ``mask_mod`` / ``OnlineFunc`` definitions) and calls it the way a model does: ``mod(q, k, v)``
for prefill and decode, the autograd edge for training, ``mod(q, q_pe, kv, k_pe)`` and the paged call form for
latent-attention decode.  ``listed()`` names twelve points; ``draw()`` takes more from the same ranges (``KINDS``).
"""
import functools
import math

import torch

import attentionengine_amd  # noqa: F401  (puts attn_engine, core and attn_script on the path)
import attn_script
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
PAGE = 64              # tokens per page of the paged latent cache
LATENT, ROPE = 512, 64  # columns of the latent cache and of its rope part


def _case(name, kind, dtype, batch, heads, heads_kv, seq_q, seq_kv, dim, dim_v, **more):
    case = {"name": name, "kind": kind, "dtype": dtype, "batch": batch, "heads": heads, "heads_kv": heads_kv,
            "seq_q": seq_q, "seq_kv": seq_kv, "dim": dim, "dim_v": dim_v}
    case.update(more)
    return case


def listed():
    return [
        # One user's short prompt in a grouped-query model, layer by layer: launch and latency bound.
        _case("prompt_short", "prompt", "bf16", 1, 32, 8, 333, 333, 128, 128),
        # The benchmark's causal prefill: two sequences of 4096 tokens.
        _case("prefill_causal_4k", "prefill", "fp16", 2, 32, 32, 4096, 4096, 128, 128),
        # Prefill of a latent-attention model before its up-projections are absorbed: 192 / 128 columns, 128 heads.
        _case("prefill_192_128", "prefill_wide_key", "bf16", 1, 128, 128, 2500, 2500, 192, 128),
        # A batch of padded documents through a bidirectional encoder of narrow heads.
        _case("encoder_ragged", "encoder", "bf16", 16, 16, 16, 1000, 1000, 64, 64),
        # The benchmark's sigmoid attention (no mask, scalar bias as a custom input).
        _case("sigmoid_4k", "sigmoid", "fp16", 2, 32, 32, 4096, 4096, 128, 128),
        # Long documents under a sliding window, the mask given as a mask_mod.
        _case("window_256", "window", "fp16", 2, 32, 32, 4096, 4096, 128, 128, window=256),
        # One attention layer of a training step: forward, then dq, dk and dv.
        _case("train_causal_2k", "train", "bf16", 4, 32, 32, 2048, 2048, 128, 128),
        # One token of one conversation against its cache (the decode script's shape): latency bound.
        _case("gqa_decode_b1", "gqa_decode", "fp16", 1, 32, 8, 1, 8192, 128, 128),
        # The same step of a server that has 64 conversations in flight, cache length not a multiple of any tile.
        _case("gqa_decode_b64", "gqa_decode_batch", "fp16", 64, 32, 8, 1, 8001, 128, 128),
        # Latent-attention decode, full batch: the benchmark's shape.
        _case("mla_decode_b128", "mla_decode", "bf16", 128, 128, 1, 1, 4096, LATENT + ROPE, LATENT),
        # Latent-attention decode through a paged cache whose entries have very different lengths.
        _case("mla_paged_b8", "mla_paged", "bf16", 8, 128, 1, 1, 2048, LATENT + ROPE, LATENT),
        # A chunk of query tokens against a long cache, split over the cache and merged (the MHA inference script).
        _case("mha_decode_chunk", "mha_decode", "fp16", 1, 32, 32, 128, 8192, 128, 128),
    ]


def _log(rng, lo, hi):
    """A whole number, spread evenly over the logarithm of its range."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(sorted(KINDS))
    dtype = rng.choice(("fp16", "bf16"))
    if kind == "prompt":
        heads, kv = rng.choice(((32, 8), (32, 32), (16, 2), (16, 16), (64, 8)))
        s, d = _log(rng, 16, 2048), rng.choice((64, 128))
        return _case("", kind, dtype, rng.randint(1, 4), heads, kv, s, s, d, d)
    if kind == "prefill":
        heads, kv = rng.choice(((32, 8), (32, 32), (16, 16)))
        s, d = _log(rng, 1024, 16384), rng.choice((64, 128))
        return _case("", kind, dtype, rng.randint(1, 4), heads, kv, s, s, d, d)
    if kind == "prefill_wide_key":
        s, heads = _log(rng, 256, 8192), rng.choice((16, 32, 128))
        return _case("", kind, dtype, rng.randint(1, 4), heads, heads, s, s, 192, 128)
    if kind == "encoder":
        s, d = _log(rng, 64, 4096), rng.choice((64, 128))
        heads = rng.choice((8, 16, 32))
        return _case("", kind, dtype, _log(rng, 1, 32), heads, heads, s, s, d, d)
    if kind == "sigmoid":
        s, d, heads = _log(rng, 256, 8192), rng.choice((64, 128)), rng.choice((8, 16, 32))
        return _case("", kind, dtype, rng.randint(1, 4), heads, heads, s, s, d, d)
    if kind == "window":
        s, d, heads = _log(rng, 512, 8192), rng.choice((64, 128)), rng.choice((16, 32))
        return _case("", kind, dtype, rng.randint(1, 4), heads, heads, s, s, d, d, window=_log(rng, 64, 1024))
    if kind == "train":
        heads, kv = rng.choice(((32, 8), (32, 32), (16, 16)))
        s, d = _log(rng, 128, 8192), rng.choice((64, 128))
        return _case("", kind, dtype, rng.randint(1, 8), heads, kv, s, s, d, d)
    if kind == "gqa_decode":
        heads, kv = rng.choice(((32, 8), (16, 2), (64, 8), (32, 4)))
        return _case("", kind, dtype, rng.randint(1, 4), heads, kv, 1, _log(rng, 128, 32768), 128, 128)
    if kind == "gqa_decode_batch":
        heads, kv = rng.choice(((32, 8), (16, 2), (64, 8), (32, 4)))
        return _case("", kind, dtype, _log(rng, 8, 128), heads, kv, 1, _log(rng, 256, 16384), 128, 128)
    if kind == "mla_decode":
        return _case("", kind, dtype, _log(rng, 1, 128), rng.choice((16, 64, 128)), 1, 1, _log(rng, 256, 8192),
                     LATENT + ROPE, LATENT)
    if kind == "mla_paged":
        return _case("", kind, dtype, _log(rng, 1, 64), rng.choice((16, 64, 128)), 1, 1,
                     PAGE * _log(rng, 4, 128), LATENT + ROPE, LATENT)
    heads = rng.choice((8, 16, 32))
    return _case("", "mha_decode", dtype, rng.randint(1, 8), heads, heads, _log(rng, 1, 256), _log(rng, 512, 16384),
                 128, 128)


def draw(rng):
    top = max(_cost(c) for c in listed())
    while True:
        case = _draw_once(rng)
        if _cost(case) <= top:
            del case["name"]
            return case


def _cost(case):
    """Seconds at a plain rate of bytes and operations: orders the cases, no more."""
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 7e14


# ---- the engine of a layer type, kept as a program keeps it -------------------------------------------------------
def _mask_mod(case):
    if case["kind"] in ("prompt", "prefill", "prefill_wide_key", "train"):
        return attn_script.causal_mask
    if case["kind"] == "window":
        return attn_script.make_sliding_window_mask(case["window"])
    return None


@functools.lru_cache(maxsize=64)
def _engine_of(items):
    case = dict(items)
    dt = DTYPES[case["dtype"]]
    b, h, hkv = case["batch"], case["heads"], case["heads_kv"]
    meta = (meta_tensor(b, h, case["seq_q"], case["dim"], dtype=dt),
            meta_tensor(b, hkv, case["seq_kv"], case["dim"], dtype=dt),
            meta_tensor(b, hkv, case["seq_kv"], case["dim_v"], dtype=dt))
    if case["kind"] == "sigmoid":
        return AttentionEngine(meta, CustomIO({"softmax_bias": (1,)}),
                               attn_script.make_sigmoid_score_mod(1 / math.sqrt(case["dim"])), None,
                               attn_script.OnlineIdentity())
    # the latent cache is scored with the scale of the 128 + 64 columns it stands for
    scale = 1 / math.sqrt(192) if case["kind"] in ("mla_decode", "mla_paged") else 1 / math.sqrt(case["dim"])
    more = {"kv_shared": True} if case["kind"] in ("mla_decode", "mla_paged") else {}
    if case["kind"] == "mla_paged":
        more["backend"] = "cute"       # the call form that takes a paged cache and returns (out, lse)
    return AttentionEngine(meta, CustomIO({}), attn_script.make_scale_score_mod(scale), _mask_mod(case),
                           attn_script.OnlineSoftmax(), **more)


def _engine(case):
    return _engine_of(tuple(sorted((k, v) for k, v in case.items() if k != "name")))


# ---- inputs --------------------------------------------------------------------------------------------------------
def _lengths(case):
    """Cached tokens of every entry of a paged batch: spread evenly from one token to the whole table."""
    n, top = case["batch"], case["seq_kv"]
    return [max(1, (i + 1) * top // n - (i * 7) % PAGE) for i in range(n)]


def prepare(case, seed):
    dt = DTYPES[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dt)
    b, h, hkv, sq, skv = case["batch"], case["heads"], case["heads_kv"], case["seq_q"], case["seq_kv"]
    state = {"kind": case["kind"], "mod": _engine(case)}
    if case["kind"] == "mla_decode":
        state["args"] = (normal(b, 1, h, LATENT), normal(b, 1, h, ROPE), normal(b, skv, 1, LATENT), normal(b, skv, 1, ROPE))
        return state
    if case["kind"] == "mla_paged":
        per_entry = skv // PAGE
        order = torch.randperm(b, generator=g, device="cuda")
        lengths = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")[order].contiguous()
        pages = torch.randperm(b * per_entry, generator=g, device="cuda").to(torch.int32).view(b, per_entry)
        state["args"] = (normal(b, 1, h, LATENT + ROPE), normal(b * per_entry, PAGE, 1, LATENT + ROPE))
        state["pages"] = {"block_table": pages, "cache_seqlens": lengths}
        return state
    q, k, v = normal(b, sq, h, case["dim"]), normal(b, skv, hkv, case["dim"]), normal(b, skv, hkv, case["dim_v"])
    if case["kind"] == "train":
        state["leaves"] = tuple(t.requires_grad_(True) for t in (q, k, v))
        state["dout"] = normal(b, sq, h, case["dim_v"])
    elif case["kind"] == "sigmoid":
        state["args"] = (q, k, v, torch.tensor([-math.log(skv)], dtype=torch.float32, device="cuda"))
    else:
        state["args"] = (q, k, v)
    return state


def run(state):
    mod = state["mod"]
    if state["kind"] == "train":
        out = mod(*state["leaves"])
        grads = torch.autograd.grad(out, state["leaves"], state["dout"])
        return (out.detach(),) + tuple(grads)
    if state["kind"] == "mla_paged":
        return mod(*state["args"], **state["pages"])
    if state["kind"] == "sigmoid":
        return mod(*state["args"])
    out, rowscales = mod.forward_with_rowscales(*state["args"])
    return {"out": out, "lse": rowscales["lse"]}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def _visible_pairs(case):
    """(query, key) pairs of one head that are not masked."""
    sq, skv = case["seq_q"], case["seq_kv"]
    if _mask_mod(case) is None:
        return sq * skv
    w = min(case.get("window", sq), sq)
    return w * (w + 1) // 2 + (sq - w) * w


def work(case):
    b, h, hkv, sq, skv, d, dv = (case[n] for n in ("batch", "heads", "heads_kv", "seq_q", "seq_kv", "dim", "dim_v"))
    if case["kind"] in ("mla_decode", "mla_paged"):
        tokens = sum(_lengths(case)) if case["kind"] == "mla_paged" else b * skv
        table = 4 * (b * skv // PAGE + b) if case["kind"] == "mla_paged" else 0
        return {"bytes": 2 * (tokens * d + b * h * (d + dv)) + 4 * b * h + table, "flops": 2 * h * tokens * (d + dv)}
    q, k, v, o = b * sq * h * d, b * skv * hkv * d, b * skv * hkv * dv, b * sq * h * dv
    pairs = b * h * _visible_pairs(case)
    if case["kind"] == "train":
        # forward: two products a pair; backward: scores and dp again, dq, dk, dv.  q, k, v, dout in, out and gradients out.
        return {"bytes": 2 * (q + k + v + o + o + q + k + v), "flops": 2 * pairs * (d + dv) + 2 * pairs * (3 * d + 2 * dv)}
    lse = 0 if case["kind"] == "sigmoid" else 4 * b * h * sq
    return {"bytes": 2 * (q + k + v + o) + lse, "flops": 2 * pairs * (d + dv)}


def tolerance(case):
    # the weights of the second product and the results are rounded to the input type; sums are fp32
    return {"rel": 3e-3 if case["dtype"] == "fp16" else 1e-2}


KINDS = {c["kind"] for c in listed()}
