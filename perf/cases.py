"""The attention calls a user of this framework makes, as cases to time and compare.

Two entry points are called, in the way a user's program calls them:

* training: `triton_flash_attention(module, query, key, value, mask, scaling)`, the function a patched
  GPT-OSS model calls once per layer, and its backward.  Tensors arrive as the model hands them over: query
  and key contiguous after the rotary embedding, value a transposed view of (B, S, G, D), dO as (B, S, H, D),
  the sink logits a parameter in the model's dtype.
* inference on a key / value cache: `attention(q, k, v, sinks, scale, window, start_q)` without gradients, with
  the new tokens at the end of the cache.

Shapes are GPT-OSS attention (64 query heads on 8 KV heads, head_dim 64, softmax scale 1/8, every other layer with
a sliding window of 128), shares of it when heads are split over GPUs, and the small 8 / 2 head problem.  q, k,
v, dO and the sink logits are N(0, 1).
"""
from __future__ import annotations

import types

import torch

from oregon_gpt_oss_patching_amd import attention, doc_start_from_position_ids, triton_flash_attention

HEAD_DIM = 64
SCALE = 0.125
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(mode, batch, queries, keys=None, window=0, dtype="bf16", heads=64, kv_heads=8, lengths="", docs=""):
    """mode: "train" (forward + backward, as many queries as keys) or "cache" (forward, the queries are the last
    of the keys).  lengths: valid length of each right-padded row.  docs: lengths of the documents packed into the row."""
    return dict(mode=mode, dtype=dtype, batch=batch, heads=heads, kv_heads=kv_heads, queries=queries,
                keys=queries if keys is None else keys, window=window, lengths=lengths, docs=docs)


def listed():
    return [
        # one new token of one sequence: the smallest call, latency and launches
        dict(_case("cache", 1, 1, 2049), name="decode_1"),
        # one new token for each sequence of a serving batch: the key / value cache is read once, nothing else matters
        dict(_case("cache", 16, 1, 8192), name="decode_16"),
        # a chunk of a long prompt behind a filled cache
        dict(_case("cache", 1, 1024, 8192), name="prefill_chunk"),
        # two short samples padded to the longest, which is any length
        dict(_case("train", 2, 383), name="short_full"),
        # the layer at the context most fine-tuning runs use, sliding-window layer
        dict(_case("train", 1, 4096, window=128), name="layer4k_window"),
        # a fine-tuning batch whose length is what its longest sample happens to have, both layer types
        dict(_case("train", 2, 3001), name="ragged_full"),
        dict(_case("train", 2, 3001, window=128), name="ragged_window"),
        # right-padded batch with the valid lengths handed over
        dict(_case("train", 4, 4096, lengths="3309,1968,1554,4079"), name="padded_full"),
        # documents packed into one row, kept apart
        dict(_case("train", 1, 8192, docs="1841,222,3067,640,95,1502,825"), name="packed_full"),
        # a model kept in float32
        dict(_case("train", 1, 1024, dtype="fp32"), name="float32_full"),
        # long context, both layer types: the largest calls
        dict(_case("train", 1, 16384), name="layer16k_full"),
        dict(_case("train", 1, 16384, window=128), name="layer16k_window"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(lo * (hi / lo) ** rng.random() + 0.5))


def draw(rng):
    """One more case: any of the uses above, sizes over their whole range (log-uniform, any residue)."""
    use = rng.choice(("decode", "prefill", "layer", "ragged", "ragged", "padded", "packed", "float32"))
    heads, kv_heads = rng.choice(((64, 8), (64, 8), (64, 8), (32, 4), (8, 1), (8, 2)))
    window = rng.choice((0, 0, 128))
    shape = dict(window=window, heads=heads, kv_heads=kv_heads)
    if use == "decode":
        batch = _log_int(rng, 1, 32)
        return _case("cache", batch, 1, _log_int(rng, 128, min(32768, 262144 // batch)), **shape)
    if use == "prefill":
        queries = _log_int(rng, 17, 2048)
        return _case("cache", 1, queries, queries + _log_int(rng, 64, 16384), **shape)
    if use == "float32":
        return _case("train", rng.randint(1, 2), _log_int(rng, 64, 1024), dtype="fp32", **shape)
    if use == "layer":                                     # lengths a program chooses: multiples of 64
        batch = rng.choice((1, 1, 2))
        return _case("train", batch, 64 * _log_int(rng, 4, 240 // batch), **shape)
    batch = 1 if use == "packed" else _log_int(rng, 1, 8)
    length = _log_int(rng, 64, 12000 // batch)
    if use == "padded":
        lengths = [rng.randint(max(1, length // 4), length) for _ in range(batch)]
        return _case("train", batch, length, lengths=",".join(map(str, lengths)), **shape)
    if use == "packed":
        docs, left = [], length
        while left > 0:
            docs.append(min(left, _log_int(rng, 32, 4096)))
            left -= docs[-1]
        return _case("train", batch, length, docs=",".join(map(str, docs)), **shape)
    return _case("train", batch, length, **shape)


def _ints(text):
    return [int(x) for x in text.split(",")] if text else []


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    b, h, kv, sq, skv = (case[x] for x in ("batch", "heads", "kv_heads", "queries", "keys"))

    def normal(*shape):
        return torch.randn(shape, generator=g, device=dev).to(dtype)

    q = normal(b, h, sq, HEAD_DIM)
    k = normal(b, kv, skv, HEAD_DIM)
    v = normal(b, skv, kv, HEAD_DIM).transpose(1, 2)
    sinks = normal(h)
    state = dict(q=q, k=k, v=v, sinks=sinks, window=case["window"] or None, start=skv - sq, mode=case["mode"])
    if case["mode"] == "train":
        state["d_out"] = normal(b, sq, h, HEAD_DIM)
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
        state["module"] = types.SimpleNamespace(sinks=torch.nn.Parameter(sinks), sliding_window=state["window"])
        state["seqlens"] = torch.tensor(_ints(case["lengths"]), dtype=torch.int32, device=dev) if case["lengths"] else None
        docs = _ints(case["docs"])
        state["position_ids"] = torch.cat([torch.arange(n) for n in docs]).view(1, -1).to(dev) if docs else None
    return state


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    if state["mode"] == "cache":
        with torch.no_grad():
            return attention(q, k, v, state["sinks"], SCALE, state["window"], state["start"])
    module, extra = state["module"], {}
    if state["seqlens"] is not None:
        extra["seqlens"] = state["seqlens"]
    if state["position_ids"] is not None:
        extra["doc_start"] = doc_start_from_position_ids(state["position_ids"])
    out, _ = triton_flash_attention(module, q, k, v, None, SCALE, **extra)
    dq, dk, dv, dsinks = torch.autograd.grad(out, (q, k, v, module.sinks), state["d_out"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv, "dsinks": dsinks}


def _pairs(first, last, window):
    """Visible (query, key) pairs of queries first .. last - 1 of one sequence that starts at key 0."""
    def upto(n):
        if not window or n <= window:
            return n * (n + 1) // 2
        return window * (window + 1) // 2 + (n - window) * window
    return upto(last) - upto(first)


def work(case):
    b, h, kv, sq, skv, window = (case[x] for x in ("batch", "heads", "kv_heads", "queries", "keys", "window"))
    elem = DTYPES[case["dtype"]].itemsize
    row = HEAD_DIM * elem
    if case["mode"] == "cache":
        seen = min(skv, sq + window - 1) if window else skv
        return {"bytes": b * row * (2 * h * sq + 2 * kv * seen) + h * elem,
                "flops": 4 * HEAD_DIM * h * b * _pairs(skv - sq, skv, window)}
    spans = _ints(case["lengths"]) or _ints(case["docs"]) or [sq] * b
    rows_in = sum(spans)
    pairs = sum(_pairs(0, n, window) for n in spans)
    # read q, k, v, dO (the rows that exist); write O, dQ, dK, dV (all rows), the sinks' gradient
    return {"bytes": row * (rows_in * (2 * h + 2 * kv) + b * sq * (2 * h + 2 * kv)) + 2 * h * elem,
            "flops": 14 * HEAD_DIM * h * pairs}


def tolerance(case):
    """Four times what the outputs differ by from the same formulas in float64: 2.1e-3 to 2.5e-3 with bf16 operands and
    results (3.2e-3 for the 64 sums of the sinks' gradient), 3.6e-7 to 1.65e-6 in float32 (dK and dV, the longest sums)."""
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 7e-6}
