"""Performance cases: the calls that a decode loop makes of this library.

Every case is one call of a public entry point of kvbridge_amd on a synthetic
cache that lies in GPU memory: one-sequence decode (short and long contexts,
the library's own launch and the reference's), several query rows per
sequence, float caches, head sizes between the powers of two, ragged batches
over a shared page pool, and the cache writer for prefill chunks and decode
steps.  Queries are N(0,1) rounded to fp16; keys and values are N(0,1),
quantised to int8 with one absmax / 127 scale per (token, kv head) unless the
case keeps a float cache; page tables are random permutations of the pool.
"""
import math

import numpy as np
import torch

import kvbridge_amd as kvb

DEVICE = "cuda"
SRC_TYPES = {"f32": (torch.float32, kvb.KVB_SRC_F32), "f16": (torch.float16, kvb.KVB_SRC_F16),
             "bf16": (torch.bfloat16, kvb.KVB_SRC_BF16)}
OUT_TYPES = {"f32": (torch.float32, kvb.KVB_OUT_F32), "f16": (torch.float16, kvb.KVB_OUT_F16)}


def _single(name, entry, rows, q_heads, kv_heads, dim, page, tokens, split, *, begin=0, cache="int8", out="f32"):
    case = {"entry": entry, "rows": rows, "q_heads": q_heads, "kv_heads": kv_heads, "dim": dim, "page": page,
            "tokens": tokens, "begin": begin, "split": split, "cache": cache, "out": out}
    return dict(case, name=name) if name else case


def _batch(name, rows, q_heads, kv_heads, dim, page, batch, shortest, longest, length_seed, split, *,
           outliers=0.0, out="f16"):
    case = {"entry": "batched", "rows": rows, "q_heads": q_heads, "kv_heads": kv_heads, "dim": dim, "page": page,
            "batch": batch, "shortest": shortest, "longest": longest, "length_seed": length_seed, "split": split,
            "outliers": outliers, "cache": "int8", "out": out}
    return dict(case, name=name) if name else case


def _append(name, tokens, kv_heads, dim, page, src, layout):
    case = {"entry": "append", "tokens": tokens, "kv_heads": kv_heads, "dim": dim, "page": page, "src": src,
            "layout": layout}
    return dict(case, name=name) if name else case


def listed():
    return [
        # A short chat turn on a small model: launch and latency are all there is.
        _single("short_512", "fused", 1, 8, 2, 64, 16, 512, 128),
        # The benchmark's call: one long sequence, single launch, fp16 output.
        _single("long_64k", "fused", 1, 32, 8, 128, 64, 65536, 2048, out="f16"),
        # The reference's own entry point (its 256-token splits) on a context of ordinary, odd length.
        _single("reference_8k", "reference", 1, 32, 8, 128, 64, 8191, 256),
        # Four query rows of one sequence (verifying drafted tokens), 16 head-rows per kv head.
        _single("four_rows_16k", "two", 4, 32, 8, 128, 64, 16001, 512),
        # The reference's dense geometry through its MMA entry point.
        _single("dense_64k", "mma", 8, 24, 4, 256, 32, 65536, 256),
        # A cache kept in fp32 (the descriptor's int8 = 0).
        _single("float_cache_8k", "two", 1, 32, 8, 128, 16, 8192, 512, cache="f32"),
        # A head size that is not a power of two, small pages.
        _single("head_dim_96_8k", "two", 1, 32, 8, 96, 16, 8000, 512),
        # Ragged serving batch over a shared pool of 64-token pages.
        _batch("ragged_batch", 1, 32, 8, 128, 64, 16, 1024, 32768, 0x4B56423, 5120),
        # Many short conversations over a pool of 16-token pages.
        _batch("small_page_batch", 1, 32, 8, 128, 16, 32, 100, 4000, 7, 512),
        # The largest: four 128K-token contexts, wide GQA, outlier tokens.
        _batch("long_batch", 1, 64, 8, 128, 64, 4, 131072, 131072, 1, 2048, outliers=0.01),
        # Writing a prefill chunk into the cache.
        _append("append_prefill_4k", 4096, 8, 128, 64, "f16", "prefill"),
        # Writing one decode step of 64 sequences into the cache.
        _append("append_step_64", 64, 8, 128, 16, "bf16", "scattered"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _split_for(tokens, splits):
    """Tokens per split, whole 64-token tiles, for about `splits` splits."""
    return max(64, -(-tokens // splits // 64) * 64)


def draw(rng):
    kind = rng.randrange(12)
    heads = rng.choice([(8, 2, 64), (32, 8, 128), (16, 4, 128), (8, 8, 128), (64, 8, 128)])
    page = rng.choice([16, 32, 64])
    if kind == 0:
        return _single("", "fused", 1, *heads, page, _log_int(rng, 64, 4096), rng.choice([64, 128, 256]),
                       out=rng.choice(["f32", "f16"]))
    if kind == 1:
        tokens = _log_int(rng, 4096, 65536)
        return _single("", "fused", 1, *heads, page, tokens, _split_for(tokens, 32), out=rng.choice(["f32", "f16"]))
    if kind == 2:
        tokens = _log_int(rng, 256, 32768)
        begin = rng.choice([0, 0, 64, rng.randrange(tokens // 2)])
        return _single("", "reference", 1, *heads, page, tokens, 256, begin=begin)
    if kind == 3:
        tokens = _log_int(rng, 512, 32768)
        return _single("", "two", rng.randint(2, 8), *rng.choice([(32, 8, 128), (64, 8, 128), (24, 4, 256)]), page,
                       tokens, rng.choice([256, 512, 1024]))
    if kind == 4:
        tokens = _log_int(rng, 1024, 65536)
        return _single("", "mma", 8, 24, 4, 256, 32, tokens, 256, begin=32 * rng.choice([0, 0, 1, 5]))
    if kind == 5:
        tokens = _log_int(rng, 128, 8192)
        return _single("", "two", rng.choice([1, 1, 2]), *rng.choice([(8, 2, 64), (32, 8, 128), (24, 4, 256)]), page,
                       tokens, rng.choice([128, 256, 512]), cache="f32")
    if kind == 6:
        tokens = _log_int(rng, 128, 8192)
        return _single("", "two", 1, *rng.choice([(32, 8), (16, 16), (24, 4)]), rng.choice([72, 80, 96, 112, 160, 192]),
                       rng.choice([16, 32, 48, 64]), tokens, rng.choice([128, 256, 512]))
    if kind == 7:
        longest = _log_int(rng, 2048, 32768)
        return _batch("", 1, *rng.choice([(32, 8, 128), (64, 8, 128), (16, 4, 128)]), 64, rng.randint(2, 16),
                      max(1, longest // 32), longest, rng.randrange(1 << 20), rng.choice([1024, 2048, 5120]),
                      out=rng.choice(["f32", "f16"]))
    if kind == 8:
        longest = _log_int(rng, 256, 4096)
        return _batch("", 1, *heads, rng.choice([16, 32]), rng.randint(2, 32), max(1, longest // 32), longest,
                      rng.randrange(1 << 20), rng.choice([256, 512]), out=rng.choice(["f32", "f16"]))
    if kind == 9:
        longest = _log_int(rng, 32768, 131072)
        return _batch("", 1, 64, 8, 128, 64, rng.randint(2, 4), longest // 2, longest, rng.randrange(1 << 20), 2048,
                      outliers=0.01)
    shape = rng.choice([(2, 64), (8, 128), (4, 128), (4, 256)])
    src = rng.choice(["f32", "f16", "bf16"])
    if kind == 10:
        return _append("", _log_int(rng, 256, 16384), *shape, page, src, "prefill")
    return _append("", _log_int(rng, 1, 255), *shape, page, src, "scattered")


# ---- inputs, made from the seed alone ------------------------------------------

def _lengths(case):
    """Tokens of every sequence of a case."""
    if case["entry"] != "batched":
        return [case["tokens"]]
    return [int(t) for t in np.random.default_rng(case["length_seed"]).integers(
        case["shortest"], case["longest"], size=case["batch"], endpoint=True)]


def _rows(g, pages, kv_heads, page, dim, outliers, int8):
    """Rows of a pool, token-major: codes and scales (int8), or values and ones."""
    codes = torch.empty((pages, kv_heads, page, dim), dtype=torch.int8 if int8 else torch.float32, device=DEVICE)
    scales = torch.ones((pages, kv_heads, page), device=DEVICE)
    step = max(1, (1 << 26) // (kv_heads * page * dim))  # bounded temporaries
    for p in range(0, pages, step):
        x = torch.randn((min(step, pages - p), kv_heads, page, dim), generator=g, device=DEVICE)
        if outliers > 0:  # whole tokens at 8 times the standard deviation
            hit = torch.rand((x.shape[0], 1, page, 1), generator=g, device=DEVICE) < outliers
            x = torch.where(hit, x * 8.0, x)
        if int8:
            s = x.abs().amax(-1) / 127.0
            scales[p:p + step] = s
            codes[p:p + step] = torch.clamp(torch.round(x / s[..., None]), -127, 127).to(torch.int8)
        else:
            codes[p:p + step] = x
    return codes, scales


def _attention_inputs(case, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    lengths, page, rows = _lengths(case), case["page"], case["rows"]
    page_counts = [-(-t // page) for t in lengths]
    pages = sum(page_counts)
    t = {"q": torch.randn(len(lengths) * rows * case["q_heads"] * case["dim"], generator=g, device=DEVICE)
         .half().float()}
    int8, outliers = case["cache"] == "int8", case.get("outliers", 0.0)
    t["k"], t["ks"] = _rows(g, pages, case["kv_heads"], page, case["dim"], outliers, int8)
    v, t["vs"] = _rows(g, pages, case["kv_heads"], page, case["dim"], outliers, int8)
    t["v"] = v.transpose(2, 3).contiguous()  # the cache keeps V dim-major
    del v
    t["table"] = torch.randperm(pages, generator=g, device=DEVICE).to(torch.int32)
    as_i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEVICE)  # noqa: E731
    t["starts"] = as_i32([0] + list(np.cumsum(lengths)))
    t["offsets"] = as_i32([0] + list(np.cumsum(page_counts)[:-1]))
    t["kpos"] = torch.cat([torch.arange(n, device=DEVICE) for n in lengths])
    t["qpos"] = torch.cat([torch.arange(n - rows, n, device=DEVICE) for n in lengths])
    return t, lengths, pages


def _append_inputs(case, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    tokens, kv_heads, dim, page = case["tokens"], case["kv_heads"], case["dim"], case["page"]
    dtype = SRC_TYPES[case["src"]][0]
    prefill = case["layout"] == "prefill"
    # A prefill chunk fills consecutive slots of random pages; a decode step writes one slot of a page per sequence.
    pages = -(-tokens // page) + 1 if prefill else 2 * tokens
    order = torch.randperm(pages, generator=g, device=DEVICE)
    t = torch.arange(tokens, device=DEVICE)
    if prefill:
        t = t + page // 4 if case["tokens"] % 2 else t  # odd chunks continue a page that is partly full
        slots = order[t // page] * page + t % page
    else:
        slots = order[:tokens] * page + torch.randint(0, page, (tokens,), generator=g, device=DEVICE)
    new = [torch.randn((tokens, kv_heads, dim), generator=g, device=DEVICE).to(dtype) for _ in "kv"]
    return {"k_new": new[0], "v_new": new[1], "slots": slots.to(torch.int32)}, pages


def _pool(case, pages):
    """An empty pool: codes and scales are zero."""
    kv_heads, dim, page = case["kv_heads"], case["dim"], case["page"]
    return {"k": torch.zeros((pages, kv_heads, page, dim), dtype=torch.int8, device=DEVICE),
            "v": torch.zeros((pages, kv_heads, dim, page), dtype=torch.int8, device=DEVICE),
            "ks": torch.zeros((pages, kv_heads, page), device=DEVICE),
            "vs": torch.zeros((pages, kv_heads, page), device=DEVICE)}


def prepare(case, seed):
    state = {"entry": case["entry"]}
    if case["entry"] == "append":
        t, pages = _append_inputs(case, seed)
        state.update(t=t, pool=_pool(case, pages))
        state["shape"] = kvb.append_shape(case["tokens"], case["kv_heads"], case["dim"], case["page"], pages,
                                          SRC_TYPES[case["src"]][1])
        return state
    t, lengths, pages = _attention_inputs(case, seed)
    geometry = (case["rows"], case["q_heads"], case["kv_heads"], case["dim"], case["page"], pages)
    scale, int8 = 1.0 / math.sqrt(case["dim"]), case["cache"] == "int8"
    if case["entry"] == "batched":
        shape = kvb.make_batch_shape(len(lengths), *geometry, max(lengths), sum(lengths), pages, case["split"], scale,
                                     int8)
        inp = kvb.batch_input(t["q"], t["qpos"], t["starts"], t["offsets"], t["kpos"], t["table"], t["k"], t["v"],
                              t["ks"], t["vs"])
        scratch, scalars = kvb.batch_scratch_elements(shape), kvb.batch_output_scalar_elements(shape)
    else:
        shape = kvb.make_shape(*geometry, case["tokens"], case["begin"], case["tokens"], scale, int8)
        inp = kvb.device_input(t["q"], t["qpos"], t["kpos"], t["table"], t["k"], t["v"], t["ks"], t["vs"])
        scratch, scalars = kvb.scratch_elements(shape, case["split"]), kvb.output_scalar_elements(shape)
    dtype, out_type = OUT_TYPES[case["out"]]
    f32 = lambda n: torch.empty(n, device=DEVICE)  # noqa: E731
    state.update(t=t, shape=shape, inp=inp, split=case["split"], out_type=out_type, scratch=f32(scratch),
                 counters=torch.zeros(len(lengths) * case["kv_heads"], dtype=torch.int32, device=DEVICE),
                 m=f32(scalars), l=f32(scalars), n=f32(scalars * case["dim"]),
                 out=torch.empty(scalars * case["dim"], dtype=dtype, device=DEVICE))
    return state


def run(state):
    s, entry = state, state["entry"]
    if entry == "append":
        t, p = s["t"], s["pool"]
        kvb.append_kv(s["shape"], t["k_new"], t["v_new"], t["slots"], p["k"], p["v"], p["ks"], p["vs"])
        return p
    if entry == "fused":
        kvb.decode_attention_fused(s["shape"], s["inp"], s["split"], s["scratch"], s["counters"], s["m"], s["l"],
                                   s["n"], s["out"], s["out_type"])
    elif entry == "two":
        kvb.decode_attention(s["shape"], s["inp"], s["split"], s["scratch"], s["m"], s["l"], s["n"], s["out"],
                             s["out_type"])
    elif entry == "batched":
        kvb.decode_attention_batched(s["shape"], s["inp"], s["scratch"], s["m"], s["l"], s["n"], s["out"],
                                     s["out_type"], counters=s["counters"])
    else:
        call = kvb.launch_attention_mma if entry == "mma" else kvb.launch_attention
        call(s["shape"], s["inp"], s["scratch"], s["m"], s["l"], s["n"])
        return {"m": s["m"], "l": s["l"], "n": s["n"]}
    return {"m": s["m"], "l": s["l"], "n": s["n"], "out": s["out"]}


def work(case):
    if case["entry"] == "append":
        size = 4 if case["src"] == "f32" else 2
        rows = case["tokens"] * case["kv_heads"]
        # K and V rows in; codes and a scale each out; one slot id per token
        return {"bytes": rows * 2 * (case["dim"] * (size + 1) + 4) + 4 * case["tokens"], "flops": 0}
    lengths, dim = _lengths(case), case["dim"]
    tokens = sum(lengths) - case.get("begin", 0)
    row_heads = case["rows"] * case["q_heads"]
    kv = tokens * case["kv_heads"] * (2 * dim + 8 if case["cache"] == "int8" else 8 * dim)
    out = 0 if case["entry"] in ("reference", "mma") else (2 if case["out"] == "f16" else 4)
    outputs = len(lengths) * row_heads * (8 + dim * (4 + out))
    queries = len(lengths) * (row_heads * dim * 4 + case["rows"] * 8)
    return {"bytes": kv + tokens * 8 + 4 * (tokens // case["page"]) + queries + outputs,
            "flops": 4 * tokens * row_heads * dim}


def tolerance(case):
    if case["entry"] == "append":
        return "exact"  # integer codes; the scale is one IEEE division
    # An fp16 output is one rounding of n / l: two results that agree to 32 bits may still round apart.
    # The rest is fp32 sums over up to 131,072 tokens.
    return {"rel": 1e-3 if case["entry"] in ("fused", "two", "batched") and case["out"] == "f16" else 1e-5}


# ---- the same results in 64 bits --------------------------------------------------

def _exact_append(case, seed):
    t, pages = _append_inputs(case, seed)
    page = case["page"]
    got = {"k": None, "v": None}  # integer codes: no 64-bit value
    for name in "kv":
        scales = torch.zeros((pages, case["kv_heads"], page), dtype=torch.float64, device=DEVICE)
        slots = t["slots"].long()
        scales[slots // page, :, slots % page] = t[name + "_new"].double().abs().amax(-1) / 127.0
        got[name + "s"] = scales
    return got


def exact(case, seed):
    if case["entry"] == "append":
        return _exact_append(case, seed)
    t, lengths, _ = _attention_inputs(case, seed)
    rows, q_heads, kv_heads, dim, page = (case[k] for k in ("rows", "q_heads", "kv_heads", "dim", "page"))
    group, begin, scale = q_heads // kv_heads, case.get("begin", 0), 1.0 / math.sqrt(dim)
    q_all = t["q"].double().view(len(lengths), rows, kv_heads, group, dim)
    ms, ls, ns = [], [], []
    for b, n_tok in enumerate(lengths):
        first = int(t["offsets"][b])
        pages = t["table"][first:first + -(-n_tok // page)].long()
        start = int(t["starts"][b])
        seen = t["kpos"][start + begin:start + n_tok][None] <= t["qpos"][b * rows:(b + 1) * rows][:, None]
        seen = seen.repeat_interleave(group, 0)  # (row, head of the group) x token
        m = torch.empty((rows, kv_heads, group), dtype=torch.float64, device=DEVICE)
        l, n = torch.empty_like(m), torch.empty((rows, kv_heads, group, dim), dtype=torch.float64, device=DEVICE)
        for h in range(kv_heads):
            k = t["k"][pages, h].double() * t["ks"][pages, h].double()[..., None]
            k = k.reshape(-1, dim)[begin:n_tok]
            v = t["v"][pages, h].double() * t["vs"][pages, h].double()[:, None]
            v = v.transpose(1, 2).reshape(-1, dim)[begin:n_tok]
            score = q_all[b, :, h].reshape(rows * group, dim) @ k.T * scale
            score = score.masked_fill(~seen, -math.inf)
            top = score.amax(1, keepdim=True)
            w = torch.exp(score - torch.where(torch.isinf(top), torch.zeros_like(top), top))
            m[:, h], l[:, h] = top.view(rows, group), w.sum(1).view(rows, group)
            n[:, h] = (w @ v).view(rows, group, dim)
        ms.append(m.flatten())
        ls.append(l.flatten())
        ns.append(n.flatten())
    m, l, n = torch.cat(ms), torch.cat(ls), torch.cat(ns)
    got = {"m": m, "l": l, "n": n}
    if case["entry"] in ("fused", "two", "batched"):
        got["out"] = torch.where(l[:, None] > 0, n.view(-1, dim) / l[:, None], torch.zeros(())).flatten()
    return got
