"""Performance cases of the attention hot path, through its public entry points.

A case is a dict of plain values.  ``listed()`` names twelve; ``draw(rng)``
gives others of the same ranges.  ``kind`` says which call a case makes:

``decode``    one query per sequence over a paged cache: ``entry`` "call" is
              ``paged_decode_attention`` (``..._fp8`` for 8-bit caches), "plan"
              a prepared ``DecodeLaunch``
``verify``    ``paged_decode_attention_multi``: the last ``tokens`` of each
              sequence at once (speculative decoding)
``step``      one serving step on a cache with an 8-bit copy: the engine sets
              the lengths, ``append_tokens`` writes the new token and
              requantises the touched pages, ``paged_decode_attention_fp8``
              reads the copy
``quantize``  ``quantize_cache`` of a whole pool
``prefill``   ``prefill_attention`` over packed sequences
``chunk``     ``paged_prefill_attention``: new tokens against a paged cache
              that already holds ``prefix`` tokens of each sequence

Lengths are spread over [lo, hi] evenly in their logarithm, so a batch is as
ragged as a queue of requests; lo = hi is a uniform batch.  Values are N(0, 1)
and pages are scattered over the pool by a random permutation.
"""

import math

import torch

from flashattntile_amd import (
    DecodeLaunch,
    PagedKVCache,
    append_tokens,
    paged_decode_attention,
    paged_decode_attention_fp8,
    paged_decode_attention_multi,
    paged_prefill_attention,
    prefill_attention,
    quantize_cache,
)
from flashattntile_amd.quant import quantize_kv_pages

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_MODES = {"int8": "int8", "fp8": "float8_e4m3fn"}


def listed():
    gqa = {"heads": 32, "kv_heads": 8, "dim": 128}
    return [
        # A few short conversations, one new token each: latency and launches.
        {"name": "decode_small", "kind": "decode", "entry": "call", "dtype": "fp16", "kv": "same", "batch": 4,
         "lo": 64, "hi": 512, "page": 16, **gqa},
        # The batch the benchmark's headline runs, by an engine that prepared its launch.
        {"name": "decode_batch", "kind": "decode", "entry": "plan", "dtype": "fp16", "kv": "same", "batch": 32,
         "lo": 4096, "hi": 4096, "page": 16, **gqa},
        # One very long context.
        {"name": "decode_long", "kind": "decode", "entry": "call", "dtype": "bf16", "kv": "same", "batch": 1,
         "lo": 131072, "hi": 131072, "page": 16, **gqa},
        # Token-granular pages: an engine that shares prefixes token by token.
        {"name": "decode_page1", "kind": "decode", "entry": "plan", "dtype": "fp16", "kv": "same", "batch": 32,
         "lo": 500, "hi": 4000, "page": 1, **gqa},
        # Four drafted tokens verified per sequence of a ragged batch.
        {"name": "verify_ragged", "kind": "verify", "dtype": "bf16", "batch": 16, "lo": 1000, "hi": 8000,
         "tokens": 4, "page": 16, **gqa},
        # A full serving step of a large ragged batch on an fp8 cache.
        {"name": "step_fp8", "kind": "step", "dtype": "bf16", "kv": "fp8", "batch": 64, "lo": 500, "hi": 16000,
         "page": 16, **gqa},
        # A prefilled pool converted to 8 bits.
        {"name": "quantize_int8", "kind": "quantize", "dtype": "fp16", "kv": "int8", "pages": 8192, "page": 16,
         **gqa},
        # One short prompt: the time to its first token is what counts.
        {"name": "prefill_short", "kind": "prefill", "dtype": "fp16", "seqs": 1, "lo": 512, "hi": 512,
         "causal": True, **gqa},
        # One long prompt, the benchmark's prefill headline.
        {"name": "prefill_long", "kind": "prefill", "dtype": "bf16", "seqs": 1, "lo": 8192, "hi": 8192,
         "causal": True, **gqa},
        # A pack of prompts of different lengths.
        {"name": "prefill_pack", "kind": "prefill", "dtype": "fp16", "seqs": 8, "lo": 184, "hi": 3721,
         "causal": True, **gqa},
        # Chunked prefill: the next 512 tokens of each of 16 long prompts.
        {"name": "chunk_batch", "kind": "chunk", "dtype": "bf16", "batch": 16, "lo": 512, "hi": 512,
         "prefix": 3584, "page": 16, "causal": True, **gqa},
        # Full-precision prefill, as an evaluation or a reference run asks for.
        {"name": "prefill_fp32", "kind": "prefill", "dtype": "fp32", "seqs": 3, "lo": 300, "hi": 2000,
         "causal": True, **gqa},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "verify", "step", "quantize", "prefill", "prefill", "prefill",
                       "chunk"])
    heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 8), (8, 8), (16, 2), (64, 8), (32, 1)])
    case = {"kind": kind, "dtype": rng.choice(["fp16", "bf16"]), "heads": heads, "kv_heads": kv_heads,
            "dim": rng.choice([128, 128, 128, 64]), "page": rng.choice([16, 16, 32, 64])}
    if kind == "quantize":
        case.update(pages=_log(rng, 64, 8192), kv=rng.choice(["int8", "fp8"]), dtype=rng.choice(["fp16", "bf16"]))
        while case["pages"] * case["page"] > 8192 * 16:
            case["pages"] = case["pages"] // 2 + 1
        return case
    if kind in ("prefill", "chunk"):
        if kind == "prefill":
            case.pop("page")
            case["seqs"] = _log(rng, 1, 16)
        else:
            case["batch"] = _log(rng, 1, 16)
            case["prefix"] = _log(rng, 64, 8192)
        case["hi"] = _log(rng, 32, 8192 if kind == "prefill" else 2048)
        case["lo"] = max(1, int(case["hi"] * rng.choice([1.0, rng.uniform(0.05, 1.0)])))
        case["causal"] = kind == "chunk" or rng.random() < 0.8
        top = 4e11
        if kind == "prefill" and rng.random() < 0.25:
            case["dtype"], top = "fp32", 1.5e10
        elif rng.random() < 0.15:
            case["dim"], top = 256, 1e11
        while work(case)["flops"] > top:
            case["hi"] = case["hi"] // 2 + 1
            case["lo"] = case["lo"] // 2 + 1
        return case
    case["batch"] = _log(rng, 1, 64)
    case["hi"] = _log(rng, 64, 65536)
    case["lo"] = max(8, int(case["hi"] * rng.choice([1.0, rng.uniform(0.03, 1.0)])))
    top = 4e8
    if kind == "decode":
        case["entry"] = rng.choice(["call", "plan"])
        case["kv"] = rng.choice(["same", "same", "int8", "fp8"])
        other = rng.random()
        if other < 0.3:
            case["dim"], top = 256, 1e8
        elif other < 0.5:
            case["page"], case["kv"], top = 1, "same", 1e8
        elif other < 0.6:
            case["dtype"], case["kv"], top = "fp32", "same", 1e8
    elif kind == "verify":
        case["tokens"] = rng.choice([2, 3, 4, 8])
    else:
        case["kv"] = rng.choice(["int8", "fp8"])
    while work(case)["bytes"] > top:
        case["hi"] = case["hi"] // 2 + 8
        case["lo"] = case["lo"] // 2 + 4
    return case


def _lens(n, lo, hi):
    """``n`` lengths over [lo, hi], evenly spread in their logarithm."""
    return [int(round(lo * (hi / lo) ** ((0.5 + 0.6180339887 * i) % 1.0))) for i in range(n)]


def _causal_pairs(lq, lk, causal):
    return lq * lk - (lq * (lq - 1) // 2 if causal else 0)


def _paged(g, case, lens, dtype):
    """A cache of ``lens`` tokens whose pages are scattered over the pool."""
    page, dev = case["page"], g.device
    per = [-(-n // page) for n in lens]
    pool = sum(per) + 3
    perm = torch.randperm(pool, generator=g, device=dev).to(torch.int32)
    table = torch.zeros(len(lens), max(per), dtype=torch.int32, device=dev)
    at = 0
    for b, n in enumerate(per):
        table[b, :n] = perm[at:at + n]
        at += n
    shape = (pool, page, case["kv_heads"], case["dim"])
    k = torch.randn(shape, generator=g, device=dev, dtype=dtype)
    v = torch.randn(shape, generator=g, device=dev, dtype=dtype)
    return PagedKVCache(k, v, table, torch.tensor(lens, dtype=torch.int32, device=dev), page)


def _quantized(cache, mode):
    """The 8-bit copy of ``cache`` under the same table and lengths, and its scales."""
    qk, qv, sk, sv, _ = quantize_kv_pages(cache.k_cache, cache.v_cache, mode=_MODES[mode])
    return PagedKVCache(qk, qv, cache.page_table, cache.seq_lens, cache.page_size), {"k": sk, "v": sv}


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind, dtype = case["kind"], _DTYPES[case["dtype"]]
    heads, kv_heads, dim = case["heads"], case["kv_heads"], case["dim"]

    def randn(*shape):
        return torch.randn(shape, generator=g, device=g.device, dtype=dtype)

    if kind == "quantize":
        table = torch.randperm(case["pages"], generator=g, device=g.device).to(torch.int32).view(1, -1)
        length = torch.tensor([case["pages"] * case["page"]], dtype=torch.int32, device=g.device)
        shape = (case["pages"], case["page"], kv_heads, dim)
        return {"kind": kind, "mode": _MODES[case["kv"]],
                "cache": PagedKVCache(randn(*shape), randn(*shape), table, length, case["page"])}
    if kind == "prefill":
        lens = _lens(case["seqs"], case["lo"], case["hi"])
        cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=g.device)
        return {"kind": kind, "q": randn(sum(lens), heads, dim), "k": randn(sum(lens), kv_heads, dim),
                "v": randn(sum(lens), kv_heads, dim), "cu": cu, "longest": max(lens), "causal": case["causal"]}
    if kind == "chunk":
        lens = _lens(case["batch"], case["lo"], case["hi"])
        cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=g.device)
        return {"kind": kind, "q": randn(sum(lens), heads, dim), "cu": cu, "longest": max(lens),
                "causal": case["causal"], "cache": _paged(g, case, [n + case["prefix"] for n in lens], dtype)}
    cache = _paged(g, case, _lens(case["batch"], case["lo"], case["hi"]), dtype)
    if kind == "verify":
        return {"kind": kind, "cache": cache, "q": randn(case["batch"], case["tokens"], heads, dim)}
    q = randn(case["batch"], heads, dim)
    if kind == "step":
        # The last token of each sequence is the one the step appends.
        qcache, scales = _quantized(cache, case["kv"])
        return {"kind": kind, "q": q, "cache": cache, "qcache": qcache, "scales": scales,
                "held": cache.seq_lens - 1, "new_k": randn(case["batch"], kv_heads, dim),
                "new_v": randn(case["batch"], kv_heads, dim)}
    scales = None
    if case["kv"] != "same":
        cache, scales = _quantized(cache, case["kv"])
    state = {"kind": kind, "entry": case["entry"], "q": q, "cache": cache, "scales": scales}
    if case["entry"] == "plan":
        state["plan"] = DecodeLaunch(q, cache, scales=scales)
    return state


def run(state):
    kind = state["kind"]
    if kind == "quantize":
        qcache, scales = quantize_cache(state["cache"], mode=state["mode"])
        return {"k": qcache.k_cache, "v": qcache.v_cache, "k_scale": scales.k, "v_scale": scales.v}
    if kind == "prefill":
        return prefill_attention(state["q"], state["k"], state["v"], state["cu"], state["cu"], state["longest"],
                                 state["longest"], causal=state["causal"])
    if kind == "chunk":
        return paged_prefill_attention(state["q"], state["cache"], state["cu"], state["longest"],
                                       causal=state["causal"])
    if kind == "verify":
        return paged_decode_attention_multi(state["q"], state["cache"])
    if kind == "step":
        cache, qcache, scales = state["cache"], state["qcache"], state["scales"]
        cache.seq_lens.copy_(state["held"])  # the engine's scheduler owns the lengths
        append_tokens(cache, state["new_k"], state["new_v"], quantized=(qcache, scales))
        out = paged_decode_attention_fp8(state["q"], qcache, scales)
        return {"out": out, "seq_lens": cache.seq_lens, "k": cache.k_cache, "v": cache.v_cache,
                "qk": qcache.k_cache, "qv": qcache.v_cache, "k_scale": scales["k"], "v_scale": scales["v"]}
    if state["entry"] == "plan":
        return state["plan"].run(state["q"])
    if state["scales"] is not None:
        return paged_decode_attention_fp8(state["q"], state["cache"], state["scales"])
    return paged_decode_attention(state["q"], state["cache"])


def work(case):
    kind, heads, kv_heads, dim = case["kind"], case["heads"], case["kv_heads"], case["dim"]
    elem = 4 if case["dtype"] == "fp32" else 2
    row = kv_heads * dim
    if kind == "quantize":
        values = case["pages"] * case["page"] * row
        return {"bytes": 2 * (values * (elem + 1) + case["pages"] * kv_heads * 4), "flops": 2 * 3 * values}
    if kind == "prefill":
        lens = _lens(case["seqs"], case["lo"], case["hi"])
        return {"bytes": sum(lens) * (2 * heads + 2 * kv_heads) * dim * elem,
                "flops": sum(4 * heads * dim * _causal_pairs(n, n, case["causal"]) for n in lens)}
    lens = _lens(case["batch"], case["lo"], case["hi"])
    if kind == "chunk":
        return {"bytes": sum(2 * n * heads * dim + 2 * (n + case["prefix"]) * row for n in lens) * elem,
                "flops": sum(4 * heads * dim * _causal_pairs(n, n + case["prefix"], case["causal"])
                             for n in lens)}
    rows = case["batch"] * case.get("tokens", 1)
    kv = 2 * sum(lens) * row
    small = case.get("kv", "same") != "same"
    scales = 8 * kv_heads * sum(-(-n // case["page"]) for n in lens) if small else 0
    out = {"bytes": 2 * rows * heads * dim * elem + kv * (1 if small else elem) + scales,
           "flops": 4 * heads * dim * sum(lens) * case.get("tokens", 1)}
    if kind == "step":  # the new rows in and out, and the touched pages read and requantised
        out["bytes"] += 4 * rows * row * elem + 2 * rows * case["page"] * row * (elem + 1) + 8 * rows * kv_heads
    return out


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # About four times the measured distance from exact(): 3e-7 (fp32), 2.9e-4
    # (fp16), 1.7e-3 (bf16) and 3e-3 (bf16 queries on 8-bit codes, whose
    # dequantised values are rounded to bf16 too); fp32 sums in another order
    # over a long context differ by a little more.
    if case["dtype"] == "fp32":
        return {"rel": 4e-6}
    if case["dtype"] == "fp16":
        return {"rel": 1.2e-3}
    return {"rel": 7e-3 if case.get("kv", "same") == "same" else 1.2e-2}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v, causal):
    """q [Lq, H, D], k / v [Lk, Hkv, D]; bottom-right causal.  64 bits, a head at a time."""
    lq, heads, dim = q.shape
    lk, kv_heads = k.shape[:2]
    out = torch.empty(lq, heads, dim, dtype=torch.float64, device=q.device)
    mask = None
    if causal:
        i = torch.arange(lq, device=q.device)[:, None] + (lk - lq)
        mask = torch.arange(lk, device=q.device)[None, :] > i
    group = heads // kv_heads
    for j in range(kv_heads):
        kt = k[:, j].double().t().contiguous()
        vj = v[:, j].double()
        for h in range(j * group, (j + 1) * group):
            s = (q[:, h].double() * dim ** -0.5) @ kt
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            out[:, h] = torch.softmax(s, dim=-1) @ vj
    return out


def _tokens(cache, b, n, scales=None):
    """The first ``n`` rows of sequence ``b``: k, v [n, Hkv, D], dequantised in 64 bits where scales are given."""
    ids = cache.page_table[b, : -(-n // cache.page_size)].long()
    got = []
    for pages, name in ((cache.k_cache, "k"), (cache.v_cache, "v")):
        x = pages[ids]
        if scales is not None:
            x = x.double() * scales[name][ids].double()[:, None, :, None]
        got.append(x.reshape(-1, *x.shape[2:])[:n])
    return got


def _codes(pages, mode):
    """Codes and scales [pages, Hkv] of float pages (absmax over a page's slots and dims)."""
    top = 127.0 if mode == "int8" else 448.0
    x = pages.float()
    scale = (x.abs().amax(dim=(1, 3)) / top).clamp_min(1e-8)
    y = x / scale[:, None, :, None]
    if mode == "int8":
        return y.round().clamp(-top, top).to(torch.int8), scale
    return y.clamp(-top, top).to(torch.float8_e4m3fn), scale


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "quantize":
        cache, top = state["cache"], 127.0 if case["kv"] == "int8" else 448.0
        return {"k": None, "v": None, "k_scale": cache.k_cache.double().abs().amax(dim=(1, 3)) / top,
                "v_scale": cache.v_cache.double().abs().amax(dim=(1, 3)) / top}
    if kind in ("prefill", "chunk"):
        cu = state["cu"].tolist()
        outs = []
        for b in range(len(cu) - 1):
            lo, hi = cu[b], cu[b + 1]
            if kind == "prefill":
                k, v = state["k"][lo:hi], state["v"][lo:hi]
            else:
                k, v = _tokens(state["cache"], b, hi - lo + case["prefix"])
            outs.append(_attend(state["q"][lo:hi], k, v, case["causal"]))
        return torch.cat(outs)
    lens = _lens(case["batch"], case["lo"], case["hi"])
    cache, scales, q = state["cache"], state.get("scales"), state["q"]
    if kind == "step":
        raw, cache = cache, state["qcache"]
        for b, n in enumerate(lens):
            page, slot = int(raw.page_table[b, (n - 1) // raw.page_size]), (n - 1) % raw.page_size
            for pages, new, codes, name in ((raw.k_cache, state["new_k"], cache.k_cache, "k"),
                                            (raw.v_cache, state["new_v"], cache.v_cache, "v")):
                pages[page, slot] = new[b]
                c, s = _codes(pages[page:page + 1], case["kv"])
                codes[page:page + 1], scales[name][page:page + 1] = c, s
    outs = []
    for b, n in enumerate(lens):
        k, v = _tokens(cache, b, n, scales)
        outs.append(_attend(q[b] if q.dim() == 4 else q[b:b + 1], k, v, q.dim() == 4))
    out = torch.stack(outs) if q.dim() == 4 else torch.cat(outs)
    if kind == "step":
        return {"out": out, "seq_lens": None, "k": None, "v": None, "qk": None, "qv": None,
                "k_scale": scales["k"].double(), "v_scale": scales["v"].double()}
    return out
