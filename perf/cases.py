"""The performance cases of this repository: what its attention entry points are called with.

A case is one call (forward alone, or forward and backward) with its sizes; ``listed`` holds the
fixed ones, ``draw`` makes more from the same ranges.  ``kind`` names the entry point:

========== =====================================================================================
dense      ``ring_sliding_window_attn``            ``[batch, seq, heads, dim]``
pack       ``ring_sliding_window_attn_varlen``     ``[tokens, heads, dim]`` + ``cu_seqlens``
sink       ``ring_streaming_llm_attn``             dense, attention sinks + window
sink_pack  ``ring_streaming_llm_attn_varlen``      packed, attention sinks + window
rank       ``ring_rank_share_attn``                one context-parallel rank's chunk
rank_pack  ``ring_rank_share_attn_varlen``         the same for a chunk of a pack
merge      ``ops.merge_attn_out``                  log-sum-exp merge of two partial results
========== =====================================================================================

Inputs are N(0, 1) (projected activations after normalisation); sink keys are four times as large,
which is what makes a token a sink.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "ring-sliding-window-attention_amd"))

import ring_swa  # noqa: E402
from ring_swa.ops import merge_attn_out  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # The smallest training call: a small model's layer on one short sequence.  Launches and
        # host work are most of it.
        dict(name="dense_1k_train", kind="dense", batch=1, seq=1024, heads=4, kv_heads=4, dim=64,
             window=256, dtype="bf16", train=True, fused_qkv=False),
        # The smallest inference call: a short ragged prompt pair through a grouped-query layer.
        dict(name="dense_333_fwd", kind="dense", batch=2, seq=333, heads=8, kv_heads=2, dim=128,
             window=100, dtype="fp16", train=False, fused_qkv=False),
        # An ordinary training layer: q, k and v are slices of one fused projection, the length is
        # no multiple of anything.
        dict(name="dense_4k_train", kind="dense", batch=1, seq=4001, heads=32, kv_heads=8, dim=128,
             window=1024, dtype="bf16", train=True, fused_qkv=True),
        # Training with as many kv heads as q heads and a window far shorter than the sequence.
        dict(name="dense_8k_mha_train", kind="dense", batch=2, seq=8192, heads=32, kv_heads=32,
             dim=128, window=1000, dtype="bf16", train=True, fused_qkv=False),
        # Prefill of a long prompt: forward only.
        dict(name="dense_32k_prefill", kind="dense", batch=1, seq=32768, heads=32, kv_heads=8,
             dim=128, window=4096, dtype="bf16", train=False, fused_qkv=False),
        # Prefill of a streaming model served in batches: sinks, an odd group size (28 over 4
        # heads), head_dim 64, fp16.
        dict(name="sink_2k_fwd", kind="sink", batch=4, seq=2000, heads=28, kv_heads=4, dim=64,
             window=1000, sinks=4, impl="fused", dtype="fp16", train=False, fused_qkv=False),
        # One of eight context-parallel ranks on a 65536-token sequence, window within the
        # previous rank's chunk: the repository's headline step.
        dict(name="rank_8k_train", kind="rank", batch=1, seq=8192, heads=32, kv_heads=8, dim=128,
             window=4096, cp=8, rank=1, ring_dtypes=False, dtype="bf16", train=True),
        # The same with a window that reaches over two earlier chunks: three blocks merged into
        # the ring's fp32 / fp64 accumulators.
        dict(name="rank_4k_far_train", kind="rank", batch=1, seq=4096, heads=32, kv_heads=8,
             dim=128, window=10000, cp=8, rank=3, ring_dtypes=False, dtype="bf16", train=True),
        # One of four ranks on a pack, its chunk starting inside a sequence.
        dict(name="rank_pack_8k_train", kind="rank_pack", seq=8192, heads=32, kv_heads=8, dim=128,
             window=2048, cp=4, rank=1, shortest=64, longest=16384, pack=0, dtype="bf16",
             train=True),
        # Fine-tuning on a pack of short samples.
        dict(name="pack_16k_short_train", kind="pack", tokens=16384, heads=32, kv_heads=8, dim=128,
             window=1024, shortest=16, longest=1024, pack=1, dtype="bf16", train=True),
        # The largest call: streaming-LLM training on a long pack, four sinks per sequence.
        dict(name="sink_pack_64k_train", kind="sink_pack", tokens=65536, heads=32, kv_heads=8,
             dim=128, window=4092, sinks=4, impl="fused", shortest=8192, longest=32768, pack=2,
             dtype="bf16", train=True),
        # The merge of a ring step's partial result into the accumulators (fp32 out, fp64 lse).
        dict(name="merge_32k", kind="merge", batch=1, seq=32768, heads=32, dim=128,
             ring_dtypes=True, dtype="bf16"),
    ]


# heads / kv heads, drawn with equal odds
_HEADS = [(4, 4), (8, 2), (12, 12), (16, 4), (28, 4), (32, 8), (32, 32)]


def _spread(rng, lo, hi):
    """A whole number whose logarithm is spread evenly over [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = max((work(c) for c in listed()), key=lambda w: w["flops"])
    most_bytes = max(work(c)["bytes"] for c in listed())
    while True:
        case = _draw_any(rng)
        w = work(case)
        if w["flops"] <= most["flops"] and w["bytes"] <= most_bytes:
            return case


def _draw_any(rng):
    kind = rng.choice(["dense", "dense", "pack", "sink", "sink_pack", "rank", "rank_pack", "merge"])
    heads, kv_heads = rng.choice(_HEADS)
    dim = rng.choice([64, 128, 128])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    case = dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=dim, dtype=dtype,
                train=rng.random() < 0.7)
    if kind in ("dense", "sink"):
        case.update(batch=_spread(rng, 1, 4), seq=_spread(rng, 200, 32768),
                    window=_spread(rng, 64, 4096), fused_qkv=rng.random() < 0.3)
    elif kind in ("pack", "sink_pack"):
        tokens = _spread(rng, 2048, 65536)
        shortest = _spread(rng, 16, min(8192, tokens // 2))
        case.update(tokens=tokens, window=_spread(rng, 64, 4096), shortest=shortest,
                    longest=_spread(rng, shortest, min(32768, tokens)), pack=rng.randrange(1 << 20))
    elif kind == "rank":
        seq = _spread(rng, 1024, 8192)
        case.update(batch=1, seq=seq, window=_spread(rng, 256, 3 * seq), cp=8,
                    rank=rng.randrange(0, 8), ring_dtypes=rng.random() < 0.25)
    elif kind == "rank_pack":
        case.update(seq=_spread(rng, 1024, 8192), window=_spread(rng, 256, 4096), cp=4,
                    rank=rng.randrange(0, 4), shortest=64, longest=16384,
                    pack=rng.randrange(1 << 20))
    else:
        del case["kv_heads"], case["train"]
        case.update(batch=_spread(rng, 1, 4), seq=_spread(rng, 1024, 131072),
                    ring_dtypes=rng.random() < 0.7)
    if kind in ("sink", "sink_pack"):
        case.update(sinks=rng.choice([1, 4]), impl="split" if rng.random() < 0.2 else "fused")
    return case


# ---- sequences and visible pairs --------------------------------------------------------------
def _tokens(case):
    return case["seq"] * case["cp"] if case["kind"] == "rank_pack" else case["tokens"]


def _cu_seqlens(case):
    """The pack: lengths spread log-uniformly over [shortest, longest], the last one cut off."""
    rng, total, cu = random.Random(case["pack"]), _tokens(case), [0]
    while cu[-1] < total:
        cu.append(min(total, cu[-1] + _spread(rng, case["shortest"], case["longest"])))
    return cu


def _hops(case):
    """Earlier ranks whose chunks the rank's window reaches."""
    return min(math.ceil(case["window"] / case["seq"]), case["cp"] - 1, case["rank"])


def _pairs(n, window):
    """Visible pairs of the first ``n`` rows of a sequence: row p sees min(p, window) + 1 keys."""
    m = min(n, window + 1)
    return m * (m + 1) // 2 + (n - m) * (window + 1)


def _sink_pairs(n, window, sinks):
    """... and of its sinks that lie before the window."""
    m = max(0, n - 1 - window)
    k = min(m, sinks)
    return k * (k + 1) // 2 + sinks * (m - k)


def _visible(case):
    kind, w, sinks = case["kind"], case["window"], case.get("sinks", 0)
    if kind in ("dense", "sink"):
        return case["batch"] * (_pairs(case["seq"], w) + _sink_pairs(case["seq"], w, sinks))
    if kind == "rank":
        first = case["rank"] * case["seq"]
        return case["batch"] * (_pairs(first + case["seq"], w) - _pairs(first, w))
    cu = _cu_seqlens(case)
    lo, hi = 0, cu[-1]
    if kind == "rank_pack":
        lo, hi = case["rank"] * case["seq"], (case["rank"] + 1) * case["seq"]
    total = 0
    for a, b in zip(cu[:-1], cu[1:]):
        p, q = max(a, lo) - a, min(b, hi) - a
        if q > p:
            total += _pairs(q, w) - _pairs(p, w)
            total += _sink_pairs(q, w, sinks) - _sink_pairs(p, w, sinks)
    return total


# ---- work, tolerance, inputs and the call ------------------------------------------------------
def work(case):
    """Bytes: every tensor the caller hands over or gets back, once.  FLOPs: 4 dim per visible
    pair and q head forward, 10 dim backward."""
    d = case["dim"]
    if case["kind"] == "merge":
        rows = case["batch"] * case["seq"] * case["heads"]
        out, lse = (4, 8) if case["ring_dtypes"] else (2, 4)
        return {"bytes": rows * (d * (2 * out + 2) + 2 * lse + 4), "flops": rows * 3 * d}
    rows = case["batch"] * case["seq"] if "batch" in case else case.get("tokens", case.get("seq"))
    q_bytes = rows * case["heads"] * d * 2
    kv_bytes = 2 * rows * case["kv_heads"] * d * 2
    if case["kind"] in ("rank", "rank_pack"):
        kv_bytes *= 1 + _hops(case)
    passes = (4, 2) if case["train"] else (2, 1)  # q, out (dout, dq); k, v (dk, dv)
    return {"bytes": passes[0] * q_bytes + passes[1] * kv_bytes,
            "flops": (14 if case["train"] else 4) * d * _visible(case) * case["heads"]}


def tolerance(case):
    """Four times the largest error against the same formula in 64 bits.  16-bit probabilities and
    results: bf16 2.0e-3 to 2.9e-3 over all listed shapes (largest single value 0.09 of the rms),
    with sink keys, whose large scores make small gradients, 4.9e-3 (0.20; the split form 0.33);
    fp16 an eighth.  Merging into fp32: 5.5e-8 (1.1e-6)."""
    if case["kind"] == "merge" and case["ring_dtypes"]:
        return {"rel": 2.5e-7, "max": 5e-6}
    rel, most = (2e-2, 0.9) if case.get("sinks") else (1e-2, 0.4)
    part = 1 if case["dtype"] == "bf16" else 8
    return {"rel": rel / part, "max": most / part}


def _qkv(case, lead, normal):
    """q, k and v: tensors of their own, or slices of one fused projection's output."""
    hq, hk, d = case["heads"], case["kv_heads"], case["dim"]
    if case.get("fused_qkv"):
        x = normal(*lead, hq + 2 * hk, d)
        return x[..., :hq, :], x[..., hq:hq + hk, :], x[..., hq + hk:, :]
    return normal(*lead, hq, d), normal(*lead, hk, d), normal(*lead, hk, d)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape, dtype=dtype):
        return torch.randn(*shape, device="cuda", dtype=dtype, generator=gen)

    kind = case["kind"]
    if kind == "merge":
        b, s, h, d = (case[n] for n in ("batch", "seq", "heads", "dim"))
        ring = case["ring_dtypes"]
        return {"kind": kind,
                "out": normal(b, s, h, d, dtype=torch.float32 if ring else dtype),
                "lse": normal(b, h, s, dtype=torch.float64 if ring else torch.float32),
                "new_out": normal(b, s, h, d), "new_lse": normal(b, h, s, dtype=torch.float32)}

    lead = (case["batch"], case["seq"]) if "batch" in case else (case.get("tokens", case.get("seq")),)
    q, k, v = _qkv(case, lead, normal)
    state = {"kind": kind, "window": case["window"], "train": case["train"], "prev": []}
    sinks = case.get("sinks", 0)
    if kind in ("sink", "sink_pack"):
        state.update(sinks=sinks, impl=case["impl"])
    if kind in ("pack", "sink_pack"):
        cu = _cu_seqlens(case)
        state["cu"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
        if sinks:
            at = torch.tensor([c + j for c, e in zip(cu[:-1], cu[1:]) for j in range(min(sinks, e - c))],
                              device="cuda")
            k[at] *= 4
    elif kind == "sink":
        k[:, :sinks] *= 4
    elif kind in ("rank", "rank_pack"):
        state.update(cp=case["cp"], rank=case["rank"], ring_dtypes=case.get("ring_dtypes", False))
        hk, d = case["kv_heads"], case["dim"]
        state["prev"] = [normal(2, *lead, hk, d) for _ in range(_hops(case))]
        if kind == "rank_pack":
            state["cu"] = _cu_seqlens(case)
    if case["train"]:
        q, k, v = (t.detach().requires_grad_() for t in (q, k, v))
        state["prev"] = [t.requires_grad_() for t in state["prev"]]
        state["dout"] = normal(*lead, case["heads"], case["dim"])
    state.update(q=q, k=k, v=v)
    return state


def _forward(s):
    kind, q, k, v, w = s["kind"], s["q"], s["k"], s["v"], s["window"]
    if kind == "dense":
        return ring_swa.ring_sliding_window_attn(q, k, v, w)
    if kind == "pack":
        return ring_swa.ring_sliding_window_attn_varlen(q, k, v, w, s["cu"])
    if kind == "sink":
        return ring_swa.ring_streaming_llm_attn(q, k, v, w, num_sink_tokens=s["sinks"], impl=s["impl"])
    if kind == "sink_pack":
        return ring_swa.ring_streaming_llm_attn_varlen(q, k, v, w, s["cu"], num_sink_tokens=s["sinks"],
                                                       impl=s["impl"])
    if kind == "rank":
        return ring_swa.ring_rank_share_attn(q, k, v, s["prev"], w, s["cp"], s["rank"],
                                             ring_dtypes=s["ring_dtypes"])
    return ring_swa.ring_rank_share_attn_varlen(q, k, v, s["prev"], w, s["cu"], s["cp"], s["rank"])


def run(state):
    if state["kind"] == "merge":
        merge_attn_out(state["out"], state["lse"], state["new_out"], state["new_lse"])
        return {"out": state["out"], "lse": state["lse"]}
    if not state["train"]:
        with torch.no_grad():
            return {"out": _forward(state)}
    leaves = [state["q"], state["k"], state["v"], *state["prev"]]
    out = _forward(state)
    grads = torch.autograd.grad(out, leaves, state["dout"])
    return {"out": out.detach(), "grads": grads}
