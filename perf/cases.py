"""The calls whose speed this library is judged by, through its public entry points.

The listed cases are what a serving loop has the library do, over its range of
sizes: prefill of one small prompt, of many short ones, of long ones, with
grouped-query heads and with packed ragged lengths; decode of one sequence, of
a layer's batch, of ragged and very long contexts; the KV-cache write between
the two.  ``draw`` gives more cases of the same kinds and ranges.  Sizes are
those of the library's own benchmark, comparison suite and tests, or generic.

Query, key and value elements are N(0, 1) in fp16 (bf16 too in the cache write,
the only entry point that takes it), the scale is the default 1/sqrt(D), cache
pages are scattered over a pool by a random permutation, as a paged allocator
leaves them.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-attention-from-scratch_amd"))
import attnkernels as ak  # noqa: E402


def listed():
    return [
        # The smallest prefill of the tests and the benchmark: launch and latency only.
        {"name": "prefill_small", "kind": "prefill", "batch": 1, "heads": 4, "kv_heads": 4, "seq": 256, "dim": 64,
         "causal": False},
        # Many short prompts at once (the comparison suite's shortest shape).
        {"name": "prefill_short_batch", "kind": "prefill", "batch": 32, "heads": 16, "kv_heads": 16, "seq": 512,
         "dim": 128, "causal": True},
        # The benchmark's head size 64 shape: encoder-style attention without a mask.
        {"name": "prefill_d64", "kind": "prefill", "batch": 4, "heads": 16, "kv_heads": 16, "seq": 2048, "dim": 64,
         "causal": False},
        # One chat prompt of odd length through a grouped-query layer: a small grid.
        {"name": "prefill_prompt_gqa", "kind": "prefill", "batch": 1, "heads": 32, "kv_heads": 8, "seq": 1111,
         "dim": 128, "causal": True},
        # Packed prompts of mixed lengths through a grouped-query layer (continuous batching).
        {"name": "prefill_varlen", "kind": "varlen", "batch": 12, "heads": 32, "kv_heads": 8, "low": 64, "high": 4096,
         "lens_seed": 5, "dim": 128, "causal": True},
        # The benchmark's headline: long context, causal.
        {"name": "prefill_long", "kind": "prefill", "batch": 2, "heads": 32, "kv_heads": 32, "seq": 8192, "dim": 128,
         "causal": True},
        # One sequence's next token: the latency of an interactive decode step.
        {"name": "decode_one", "kind": "decode", "batch": 1, "heads": 32, "kv_heads": 8, "low": 1000, "high": 1000,
         "lens_seed": 0, "dim": 128, "page": 16, "partition": 0},
        # The grouped-query layer of the benchmark, a full serving batch.
        {"name": "decode_layer", "kind": "decode", "batch": 16, "heads": 32, "kv_heads": 8, "low": 8192, "high": 8192,
         "lens_seed": 0, "dim": 128, "page": 16, "partition": 0},
        # Continuous batching: ragged contexts, one query head per kv head.
        {"name": "decode_ragged", "kind": "decode", "batch": 64, "heads": 32, "kv_heads": 32, "low": 1, "high": 4096,
         "lens_seed": 0, "dim": 128, "page": 16, "partition": 0},
        # Eight query heads per kv head, ragged long contexts.
        {"name": "decode_group8", "kind": "decode", "batch": 16, "heads": 64, "kv_heads": 8, "low": 512,
         "high": 8192, "lens_seed": 3, "dim": 128, "page": 16, "partition": 0},
        # Very long contexts in many splits chosen by the caller, head size 64.
        {"name": "decode_long_d64", "kind": "decode", "batch": 8, "heads": 32, "kv_heads": 32, "low": 32768,
         "high": 32768, "lens_seed": 0, "dim": 64, "page": 16, "partition": 256},
        # The new tokens of a batch of prompts, sliced from a fused QKV projection, into the paged cache.
        {"name": "cache_write", "kind": "write", "tokens": 8192, "heads": 32, "kv_heads": 8, "dim": 128, "page": 16,
         "append": False, "dtype": "float16"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


# No drawn case costs more than the largest listed ones: the causal prefill's
# FLOP (prefill kinds) and the ragged decode's K/V bytes (decode and write).
_MOST_FLOPS = 1.0e12
_MOST_BYTES = 2.0e9


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "varlen", "decode", "decode", "decode", "write"])
    while True:
        dim = rng.choice([64, 128])
        if kind in ("prefill", "varlen"):
            kv_heads = rng.choice([4, 8, 16, 32])
            group = rng.choice([1, 1, 2, 4, 8])
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "heads": kv_heads * group, "kv_heads": kv_heads,
                    "dim": dim, "causal": rng.random() < 0.6}
            if case["heads"] > 64:
                continue
            if kind == "prefill":
                case["seq"] = _log_int(rng, 64, 8192)
            else:
                case.update(batch=max(2, case["batch"]), low=16, high=_log_int(rng, 128, 8192),
                            lens_seed=rng.randrange(1 << 20))
            if work(case)["flops"] > _MOST_FLOPS or work(case)["bytes"] > _MOST_BYTES / 4:
                continue
        elif kind == "decode":
            kv_heads = rng.choice([4, 8, 16, 32])
            group = rng.choice([1, 2, 4, 4, 8])
            high = _log_int(rng, 64, 32768)
            case = {"kind": kind, "batch": _log_int(rng, 1, 64), "heads": kv_heads * group, "kv_heads": kv_heads,
                    "low": high if rng.random() < 0.4 else max(1, high // rng.choice([2, 8, 64])), "high": high,
                    "lens_seed": rng.randrange(1 << 20), "dim": dim, "page": rng.choice([16, 16, 16, 16, 8, 32]),
                    "partition": rng.choice([0, 0, 0, 256, 512])}
            if case["heads"] > 64 or work(case)["bytes"] > _MOST_BYTES:
                continue
        else:
            case = {"kind": kind, "tokens": _log_int(rng, 1, 32768), "heads": 32, "kv_heads": rng.choice([4, 8, 32]),
                    "dim": dim, "page": rng.choice([16, 16, 16, 8, 32]), "append": rng.random() < 0.4,
                    "dtype": rng.choice(["float16", "bfloat16"])}
            if case["append"]:  # a decode step: one token per sequence
                case["tokens"] = _log_int(rng, 1, 256)
            if work(case)["bytes"] > _MOST_BYTES:
                continue
        return case


def _lens(case):
    """Sequence lengths: uniform in [low, high], the last one the longest."""
    r = random.Random(case["lens_seed"])
    return [r.randint(case["low"], case["high"]) for _ in range(case["batch"] - 1)] + [case["high"]]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float16):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def prepare(case, seed):
    g = _generator(seed)
    kind, dim = case["kind"], case["dim"]
    if kind == "prefill":
        b, n = case["batch"], case["seq"]
        s = {"q": _randn(g, b, case["heads"], n, dim), "k": _randn(g, b, case["kv_heads"], n, dim),
             "v": _randn(g, b, case["kv_heads"], n, dim)}
    elif kind == "varlen":
        lens = _lens(case)
        cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
        s = {"q": _randn(g, sum(lens), case["heads"], dim), "k": _randn(g, sum(lens), case["kv_heads"], dim),
             "v": _randn(g, sum(lens), case["kv_heads"], dim), "cu": cu, "longest": max(lens)}
    elif kind == "decode":
        lens, page = _lens(case), case["page"]
        blocks = [-(-c // page) for c in lens]
        pool = -(-sum(blocks) * 11 // 10)
        order = torch.randperm(pool, generator=g, device="cuda").to(torch.int32)
        tables = torch.zeros(len(lens), max(blocks), dtype=torch.int32, device="cuda")
        at = 0
        for i, nb in enumerate(blocks):
            tables[i, :nb] = order[at:at + nb]
            at += nb
        s = {"q": _randn(g, len(lens), case["heads"], dim), "k": _randn(g, pool, case["kv_heads"], page, dim),
             "v": _randn(g, pool, case["kv_heads"], page, dim), "tables": tables,
             "lens": torch.tensor(lens, dtype=torch.int32, device="cuda"), "longest": max(lens)}
    else:
        tokens, page, hkv = case["tokens"], case["page"], case["kv_heads"]
        dtype = getattr(torch, case["dtype"])
        qkv = _randn(g, tokens, (case["heads"] + 2 * hkv) * dim, dtype=dtype)
        key, value = qkv[:, case["heads"] * dim:].view(tokens, 2, hkv, dim).unbind(1)
        index = torch.arange(tokens, device="cuda")
        pages = tokens if case["append"] else -(-tokens // page)
        pool = -(-pages * 11 // 10)
        order = torch.randperm(pool, generator=g, device="cuda")
        rows = torch.randint(page, (tokens,), generator=g, device="cuda") if case["append"] else index % page
        slots = order[index if case["append"] else index // page] * page + rows
        s = {"key": key, "value": value, "slots": slots,
             "k": torch.zeros(pool, hkv, page, dim, dtype=dtype, device="cuda"),
             "v": torch.zeros(pool, hkv, page, dim, dtype=dtype, device="cuda")}
    return {"case": dict(case), **s}


def run(state):
    case = state["case"]
    if case["kind"] == "prefill":
        call = ak.flash_attention if case["heads"] == case["kv_heads"] else ak.flash_attention_gqa
        return call(state["q"], state["k"], state["v"], causal=case["causal"])
    if case["kind"] == "varlen":
        return ak.flash_attention_varlen(state["q"], state["k"], state["v"], state["cu"], state["longest"],
                                         causal=case["causal"])
    if case["kind"] == "decode":
        return ak.paged_decode(state["q"], state["k"], state["v"], state["tables"], state["lens"], state["longest"],
                               partition_size=case["partition"] or None)
    ak.reshape_and_cache(state["key"], state["value"], state["k"], state["v"], state["slots"])
    return state["k"], state["v"]


def work(case):
    """Bytes: each input and output element once.  FLOP: 4 n^2 D per head, half of it if causal."""
    hq, hkv, dim = case["heads"], case["kv_heads"], case["dim"]
    if case["kind"] in ("prefill", "varlen"):
        lens = [case["seq"]] * case["batch"] if case["kind"] == "prefill" else _lens(case)
        flops = sum(4.0 * hq * n * n * dim * (0.5 if case["causal"] else 1.0) for n in lens)
        return {"bytes": 2.0 * sum(lens) * dim * (2 * hq + 2 * hkv), "flops": flops}
    if case["kind"] == "decode":
        lens = _lens(case)
        pages = sum(-(-c // case["page"]) for c in lens)
        return {"bytes": 4.0 * sum(lens) * hkv * dim + 4.0 * len(lens) * hq * dim + 4.0 * (pages + len(lens)),
                "flops": 4.0 * sum(lens) * hq * dim}
    return {"bytes": 8.0 * case["tokens"] * hkv * dim + 8.0 * case["tokens"], "flops": 0.0}


def tolerance(case):
    """The cache write is a copy.  Attention rounds its probabilities and its
    output to fp16 (2^-11 each): measured, the same call with its keys permuted
    or its contexts split otherwise differs by up to 3.9e-4 (2-norm) and 2.6e-3
    (largest), and a call by up to 2.9e-4 and 5.7e-3 from float64; allowed is
    four times that."""
    if case["kind"] == "write":
        return "exact"
    return {"rel": 1.5e-3, "max": 2e-2}


def _attend(q, k, v, causal):
    """softmax(q k^T / sqrt(D) [+ causal mask]) v for one head in float64, in blocks of query rows."""
    q, kt, v = q.double(), k.double().t().contiguous(), v.double().contiguous()
    n, out = q.shape[0], torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for r in range(0, n, 2048):
        s = (q[r:r + 2048].contiguous() @ kt) * q.shape[1] ** -0.5
        if causal:
            row = torch.arange(r, r + s.shape[0], device=q.device)[:, None]
            s.masked_fill_(torch.arange(n, device=q.device)[None, :] > row, -math.inf)
        out[r:r + 2048] = torch.softmax(s, dim=1) @ v
    return out


def exact(case, seed):
    s = prepare(case, seed)
    group = case["heads"] // case["kv_heads"]
    if case["kind"] == "prefill":
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        for b in range(case["batch"]):
            for h in range(case["heads"]):
                out[b, h] = _attend(s["q"][b, h], s["k"][b, h // group], s["v"][b, h // group], case["causal"])
        return out
    if case["kind"] == "varlen":
        out, at = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda"), 0
        for n in _lens(case):
            for h in range(case["heads"]):
                out[at:at + n, h] = _attend(s["q"][at:at + n, h], s["k"][at:at + n, h // group],
                                            s["v"][at:at + n, h // group], case["causal"])
            at += n
        return out
    if case["kind"] == "decode":
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        for b, n in enumerate(_lens(case)):
            pages = s["tables"][b, :-(-n // case["page"])].long()
            for h in range(case["kv_heads"]):
                heads = slice(h * group, (h + 1) * group)
                k, v = (s[x][pages, h].reshape(-1, case["dim"])[:n] for x in ("k", "v"))
                p = (s["q"][b, heads].double() @ k.double().t().contiguous()) * case["dim"] ** -0.5
                out[b, heads] = torch.softmax(p, dim=1) @ v.double()
        return out
    page, row = s["slots"] // case["page"], s["slots"] % case["page"]
    caches = []
    for cache, new in ((s["k"], s["key"]), (s["v"], s["value"])):
        cache = cache.double()
        cache[page, :, row, :] = new.double()
        caches.append(cache)
    return tuple(caches)
