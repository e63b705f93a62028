"""Performance cases: the calls a program makes into this framework, with their sizes, inputs and tolerances.

Each case is a plain dict.  ``listed()`` gives the named ones, ``draw(rng)``
another of the same ranges, ``prepare(case, seed)`` what the program holds
before the call, ``run(state)`` one pass through the public entry points,
``work(case)`` the bytes and operations of a pass, ``exact(case, seed)`` its
result in 64 bits and ``tolerance(case)`` what two correct implementations at
the same precision may differ by.

Kinds:
  decode   ops.fog_decode: one query per sequence over a paged KV pool
  layer    KeSSieAttentionImpl.forward over a few layers of one engine step
           (K/V write, fog bias of the step, decode rows and prompt chunks)
  prefill  ops.fog_prefill: a chunk of queries at the end of a paged context
  dense    KeSSieKernels.fused_fog_attention / windowed_attention, fp16 [B,H,N,D]
  remap    ops.rope_remap_paged: recalled K moved to new positions, in place
  inject   ops.page_insert with the remap: recalled K/V from a staging buffer
  evict    ops.page_evict_compact and ops.page_gather of the survivors
  index    ops.index_query: the conversation index, similarities and top-k
"""
from __future__ import annotations

import math

import torch

from kessie_amd import ops
from kessie_amd.kessie_attention import KESSIE_STATE, KeSSieAttentionImpl, KeSSieAttentionMetadata
from kessie_amd.kessie_hip_ctypes import KeSSieKernels

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_ES = {"bf16": 2, "fp16": 2, "fp32": 4}

# Attention geometries (query heads, kv heads, head_dim): GQA ratios 1 to 16,
# the group of three that the prefill tests hold, tensor-parallel shares of
# larger models, and head_dim 64.
_GEOMS = [(32, 8, 128), (32, 8, 128), (16, 8, 128), (64, 8, 128), (32, 4, 128), (16, 1, 128), (8, 8, 128),
          (24, 8, 128), (32, 8, 64), (8, 8, 64)]

_MAX_KV_BYTES = 8.6e9    # the largest listed context
_MAX_FLOPS = 4.3e12      # the largest listed chunk


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # One short conversation in fp32, the precision the reference's CPU path runs in: the smallest
        # decode step, where launches and latency count.
        dict(name="decode_4k_fp32", kind="decode", dtype="fp32", batch=1, hq=32, hkv=8, d=128, ctx=4096, spread=1.0,
             page=16, window=0, fog="vscale", layout="native"),
        # Long-context serving: sixteen conversations of 131,072 tokens.
        dict(name="decode_128k_b16", kind="decode", dtype="bf16", batch=16, hq=32, hkv=8, d=128, ctx=131072,
             spread=1.0, page=16, window=0, fog="vscale", layout="native"),
        # A sliding-window model in fp16 on 32-token blocks: contexts of up to 32,000 tokens of which
        # the last 4,096 are seen.
        dict(name="decode_window_fp16", kind="decode", dtype="fp16", batch=12, hq=64, hkv=8, d=128, ctx=32003,
             spread=0.25, page=32, window=4096, fog="bias", layout="kv_first"),
        # One engine step of ordinary serving, decode only: 24 conversations of mixed length.
        dict(name="layer_decode", kind="layer", dtype="bf16", hq=32, hkv=8, d=128, page=16, layers=4, decode=24,
             ctx=16384, spread=0.03, prompts=0, chunk=0, prior=0, window=0, layout="block_kv"),
        # One engine step with prompts arriving among running conversations, on a head_dim 64 model.
        dict(name="layer_mixed_d64", kind="layer", dtype="bf16", hq=32, hkv=8, d=64, page=16, layers=2, decode=12,
             ctx=6000, spread=0.1, prompts=4, chunk=1111, prior=700, window=0, layout="block_kv"),
        # A chunk of a long prompt: 2,048 queries at the end of 131,072 tokens.
        dict(name="prefill_2k_on_128k", kind="prefill", dtype="bf16", batch=1, hq=32, hkv=8, d=128, chunk=2048,
             ctx=131072, page=16, window=0, fog="vscale", layout="native"),
        # The dense operator on a long sequence: 8,192 positions, 32 heads.
        dict(name="dense_fog_8k", kind="dense", batch=1, heads=32, n=8192, d=128, window=0, causal=True, fog=True),
        # The dense operator on an odd length, head_dim 64, with a window.
        dict(name="dense_window_1537", kind="dense", batch=2, heads=8, n=1537, d=64, window=1024, causal=True,
             fog=False),
        # Recalled K re-rotated in its pages.
        dict(name="remap_65k", kind="remap", dtype="bf16", tokens=65536, hkv=8, d=128, page=16, layout="native",
             theta=500000.0),
        # A recalled passage written into freshly allocated pages, K remapped on the way; the last page partly filled.
        dict(name="inject_9k", kind="inject", dtype="bf16", tokens=9005, hkv=8, d=128, page=16, layout="native",
             theta=500000.0),
        # Memory pressure: the lowest quarter of 65,536 scored pages evicted, 64 tables compacted, survivors gathered.
        dict(name="evict_gather_65k", kind="evict", dtype="bf16", seqs=64, width=1024, spare=0, hkv=8, d=128, page=16),
        # A conversation index searched with one query.
        dict(name="index_78k", kind="index", dtype="fp32", rows=78125, d=256, top_k=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "layer", "layer", "prefill", "prefill", "dense", "dense", "remap",
                       "inject", "evict", "index"])
    hq, hkv, d = rng.choice(_GEOMS)
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    page = rng.choice([16, 16, 32])
    layout = rng.choice(["native", "kv_first", "block_kv"])
    window = rng.choice([0, 0, 1024, 4096])
    fog = rng.choice(["vscale", "bias", "none"])
    while True:
        if kind == "decode":
            c = dict(kind=kind, dtype=dtype, batch=_log(rng, 1, 64), hq=hq, hkv=hkv, d=d, ctx=_log(rng, 256, 131072),
                     spread=round(rng.choice([1.0, rng.uniform(0.03, 1.0)]), 3), page=page, window=window, fog=fog,
                     layout=layout)
            if d == 128 and hq // hkv in (1, 2, 4) and rng.random() < 0.15:
                c["dtype"] = "fp32"
        elif kind == "layer":
            prompts = rng.choice([0, 0, 1, 2, 5])
            c = dict(kind=kind, dtype=dtype, hq=hq, hkv=hkv, d=d, page=page, layers=2, decode=_log(rng, 1, 48),
                     ctx=_log(rng, 512, 16384), spread=round(rng.uniform(0.03, 1.0), 3), prompts=prompts,
                     chunk=_log(rng, 24, 2048) if prompts else 0, prior=rng.choice([0, _log(rng, 16, 4096)]) if prompts else 0,
                     window=window, layout=rng.choice(["kv_first", "block_kv"]))
        elif kind == "prefill":
            chunk = _log(rng, 17, 4096)
            c = dict(kind=kind, dtype=dtype, batch=rng.choice([1, 1, 2, 4]), hq=hq, hkv=hkv, d=d, chunk=chunk,
                     ctx=max(chunk, _log(rng, 64, 131072)), page=page, window=window, fog=fog, layout=layout)
        elif kind == "dense":
            c = dict(kind=kind, batch=rng.choice([1, 1, 2, 4]), heads=rng.choice([8, 12, 16, 32]), n=_log(rng, 128, 8192),
                     d=rng.choice([64, 128]), window=rng.choice([0, 0, 1024]), causal=rng.random() < 0.8,
                     fog=rng.random() < 0.5)
        elif kind in ("remap", "inject"):
            c = dict(kind=kind, dtype=dtype, tokens=_log(rng, 64, 65536), hkv=rng.choice([8, 8, 4]), d=d, page=page,
                     layout=layout, theta=rng.choice([10000.0, 500000.0]))
        elif kind == "evict":
            c = dict(kind=kind, dtype=dtype, seqs=_log(rng, 1, 64), width=_log(rng, 16, 1024), spare=_log(rng, 1, 2000),
                     hkv=8, d=d, page=16)
        else:
            c = dict(kind=kind, dtype=rng.choice(["fp32", "fp32", "bf16"]), rows=_log(rng, 200, 300000), d=256,
                     top_k=rng.choice([3, 5, 10]))
        w = work(c)
        if w["bytes"] <= _MAX_KV_BYTES and w["flops"] <= _MAX_FLOPS and _state_bytes(c) <= 1.2e10:
            return c


# ---------------------------------------------------------------------------
# Sizes
# ---------------------------------------------------------------------------
def _lens(n, longest, spread):
    """n lengths from longest * spread to longest (spaced evenly over their logarithm), in a mixed order."""
    lo = max(1, int(longest * spread))
    if n == 1 or lo >= longest:
        return [longest] * n
    v = [int(round(math.exp(math.log(lo) + (math.log(longest) - math.log(lo)) * i / (n - 1)))) for i in range(n)]
    return [v[(i * 7 + 3) % n] if math.gcd(7, n) == 1 else v[i] for i in range(n)]


def _seqs(case):
    """(query rows, context length) of each sequence of a decode, prefill or layer case."""
    k = case["kind"]
    if k == "decode":
        return [(1, n) for n in _lens(case["batch"], case["ctx"], case["spread"])]
    if k == "prefill":
        return [(case["chunk"], case["ctx"])] * case["batch"]
    rows = [(1, n) for n in _lens(case["decode"], case["ctx"], case["spread"])]
    for i in range(case["prompts"]):  # each prompt's chunk shorter than the one before, every other one fresh
        c = max(2, case["chunk"] * (case["prompts"] - i) // case["prompts"])
        rows.append((c, c + (case["prior"] if i % 2 == 0 else 0)))
    return rows


def _pairs(rows, ctx, window):
    """Visible (query, key) pairs of `rows` causal queries at the end of ctx tokens."""
    if not window or window >= ctx:
        return rows * (ctx - rows) + rows * (rows + 1) // 2
    return sum(min(window, p + 1) for p in range(ctx - rows, ctx))


def _keys(rows, ctx, window):
    return ctx if not window else min(ctx, window + rows - 1)


def _state_bytes(case):
    if case["kind"] in ("decode", "layer", "prefill"):
        per = 2 * case["hkv"] * case["d"] * _ES[case["dtype"]]
        return sum(n for _, n in _seqs(case)) * per * case.get("layers", 1)
    return 0


def work(case):
    k = case["kind"]
    if k in ("decode", "layer", "prefill"):
        es, w, per = _ES[case["dtype"]], case["window"], 2 * case["hkv"] * case["d"] * _ES[case["dtype"]]
        b = f = 0
        for rows, ctx in _seqs(case):
            keys = _keys(rows, ctx, w)
            b += keys * per + 2 * rows * case["hq"] * case["d"] * es + 4 * -(-keys // case["page"])
            b += 4 * keys if case.get("fog", "bias") == "bias" else 0
            b += 2 * rows * per if k == "layer" else 0  # new K/V rows, read and written
            f += 4 * case["d"] * case["hq"] * _pairs(rows, ctx, w)
        if case.get("fog") == "vscale":
            b += 4 * case["ctx"]
        n = case.get("layers", 1)
        return {"bytes": b * n, "flops": f * n}
    if k == "dense":
        n, bh = case["n"], case["batch"] * case["heads"]
        pairs = _pairs(n, n, case["window"]) if case["causal"] or case["window"] else n * n
        return {"bytes": 4 * bh * n * case["d"] * 2 + 4 * n * case["fog"], "flops": 4 * case["d"] * bh * pairs}
    if k == "remap":
        return {"bytes": case["tokens"] * (2 * case["hkv"] * case["d"] * _ES[case["dtype"]] + 8), "flops": 0}
    if k == "inject":
        return {"bytes": case["tokens"] * (4 * case["hkv"] * case["d"] * _ES[case["dtype"]] + 8), "flops": 0}
    if k == "evict":
        n = case["seqs"] * case["width"]
        keep = n - n // 4
        page = case["page"] * 2 * case["hkv"] * case["d"] * _ES[case["dtype"]]
        return {"bytes": 2 * keep * page + 17 * n, "flops": 0}
    return {"bytes": case["rows"] * (case["d"] * _ES[case["dtype"]] + 4), "flops": 2 * case["rows"] * case["d"]}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=_DT[dtype])


def _pool_shape(layout, n, page, hkv, d):
    return {"native": (n, page, 2, hkv, d), "kv_first": (2, n, page, hkv, d), "block_kv": (n, 2, page, hkv, d)}[layout]


def _kv(pool, layout):
    """K and V views [pages, page, heads, head_dim] of a pool."""
    if layout == "native":
        return pool[:, :, 0], pool[:, :, 1]
    return (pool[0], pool[1]) if layout == "kv_first" else (pool[:, 0], pool[:, 1])


def _fog_weights(n):
    """The V weights of the reference's defaults: sqrt ramp over the older half, 1 after it."""
    w = torch.ones(n, dtype=torch.float32, device="cuda")
    c = n // 2
    w[:c] = (torch.arange(c, dtype=torch.float32, device="cuda") / max(c - 1, 1)).sqrt()
    return w


def _fog_bias(n, dtype=torch.float32):
    """The logit bias of the reference's defaults, in its order of operations and in `dtype`."""
    b = torch.zeros(n, dtype=dtype, device="cuda")
    c = int(n * 0.5)
    if c > 0:
        t = 1.0 - torch.arange(c, dtype=dtype, device="cuda") / c
        t.mul_(t)
        t.mul_(-0.5)
        b[:c] = t
    return b


def _recall(longest):
    return [p for p in range(11, longest, 997)][:64]


def _tables(g, seqs, page):
    """Random page tables for the sequences, over a pool with a few pages more than they use."""
    need = [-(-ctx // page) for _, ctx in seqs]
    total, width = sum(need), max(need)
    perm = torch.randperm(total + total // 16 + 1, generator=g, device="cuda")[:total].to(torch.int32)
    table = torch.zeros(len(seqs), width, dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    return table, total + total // 16 + 1


def _positions(g, tokens):
    orig = torch.randint(0, 1_000_000, (tokens,), generator=g, device="cuda", dtype=torch.int32)
    base = int(torch.randint(0, 500_000, (1,), generator=g, device="cuda"))
    return orig, torch.arange(base, base + tokens, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    k, g = case["kind"], _gen(seed)
    s = dict(case=case)
    if k in ("decode", "prefill"):
        seqs = _seqs(case)
        s["table"], pages = _tables(g, seqs, case["page"])
        s["pool"] = _randn(g, _pool_shape(case["layout"], pages, case["page"], case["hkv"], case["d"]), case["dtype"])
        rows = (case["batch"],) if k == "decode" else (case["batch"], case["chunk"])
        s["q"] = _randn(g, rows + (case["hq"], case["d"]), case["dtype"])
        s["lens"] = torch.tensor([n for _, n in seqs], dtype=torch.int32, device="cuda")
        s["max_ctx"] = max(n for _, n in seqs)
        s["vscale"] = _fog_weights(s["max_ctx"]) if case["fog"] == "vscale" else None
        s["bias"] = torch.zeros(case["batch"], s["max_ctx"], device="cuda") if case["fog"] == "bias" else None
        if s["bias"] is not None:
            for i, (_, n) in enumerate(seqs):
                s["bias"][i, :n] = _fog_bias(n)
    elif k == "layer":
        seqs = _seqs(case)
        table, pages = _tables(g, seqs, case["page"])
        hq, hkv, d, tokens = case["hq"], case["hkv"], case["d"], sum(r for r, _ in seqs)
        shape = _pool_shape(case["layout"], pages, case["page"], hkv, d)
        s["caches"] = [_randn(g, shape, case["dtype"]) for _ in range(case["layers"])]
        s["q"] = [_randn(g, (tokens, hq, d), case["dtype"]) for _ in range(case["layers"])]
        s["k"] = [_randn(g, (tokens, hkv, d), case["dtype"]) for _ in range(case["layers"])]
        s["v"] = [_randn(g, (tokens, hkv, d), case["dtype"]) for _ in range(case["layers"])]
        starts, slots = [0], []
        for i, (r, n) in enumerate(seqs):
            p = torch.arange(n - r, n, device="cuda")
            slots.append(table[i].long()[p // case["page"]] * case["page"] + p % case["page"])
            starts.append(starts[-1] + r)
        qsl = torch.tensor(starts, dtype=torch.int32)
        lens = torch.tensor([n for _, n in seqs], dtype=torch.int32)
        s["meta"] = KeSSieAttentionMetadata(
            num_actual_tokens=tokens, max_query_len=max(r for r, _ in seqs), query_start_loc=qsl.cuda(),
            max_seq_len=int(lens.max()), seq_lens=lens.cuda(), block_table=table, slot_mapping=torch.cat(slots),
            query_start_loc_cpu=qsl, seq_lens_cpu=lens)
        s["impl"] = KeSSieAttentionImpl(hq, d, d ** -0.5, hkv, sliding_window=case["window"] or None)
        s["recall"] = _recall(int(lens.max()))
    elif k == "dense":
        shape = (case["batch"], case["heads"], case["n"], case["d"])
        s["q"], s["k"], s["v"] = (_randn(g, shape, "fp16") for _ in range(3))
        s["w"] = _fog_weights(case["n"])
        s["kernels"], s["stream"] = KeSSieKernels(), torch.cuda.current_stream()
    elif k in ("remap", "inject"):
        n = -(-case["tokens"] // case["page"])
        s["pages"] = torch.randperm(n + n // 16 + 1, generator=g, device="cuda")[:n].to(torch.int32)
        pages = n + n // 16 + 1
        s["pool"] = _randn(g, _pool_shape(case["layout"], pages, case["page"], case["hkv"], case["d"]), case["dtype"])
        s["orig"], s["tgt"] = _positions(g, case["tokens"])
        if k == "inject":
            shape = (case["tokens"], case["hkv"], case["d"])
            s["new_k"], s["new_v"] = _randn(g, shape, case["dtype"]), _randn(g, shape, case["dtype"])
            s["valid"] = torch.zeros(pages, dtype=torch.int8, device="cuda")
            s["positions"] = torch.zeros(pages, dtype=torch.int32, device="cuda")
    elif k == "evict":
        n = case["seqs"] * case["width"]
        pages = n + case["spare"]
        perm = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)
        s["tables"] = perm[:n].view(case["seqs"], case["width"]).contiguous()
        s["lens"] = torch.full((case["seqs"],), case["width"], dtype=torch.int32, device="cuda")
        s["valid"] = torch.zeros(pages, dtype=torch.int8, device="cuda")
        s["valid"][perm[:n].long()] = 1
        s["scores"] = torch.rand(pages, generator=g, device="cuda")
        s["pool"] = _randn(g, (pages, case["page"], 2, case["hkv"], case["d"]), case["dtype"])
        s["staging"] = torch.empty((n - n // 4,) + tuple(s["pool"].shape[1:]), dtype=_DT[case["dtype"]], device="cuda")
    else:
        s["embeds"] = _randn(g, (case["rows"], case["d"]), case["dtype"])
        s["query"] = torch.randn(case["d"], generator=g, device="cuda")
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    c = s["case"]
    k = c["kind"]
    if k in ("decode", "prefill"):
        fn = ops.fog_decode if k == "decode" else ops.fog_prefill
        return fn(s["q"], s["pool"], s["table"], s["lens"], s["max_ctx"], fog_vscale=s["vscale"], fog_bias=s["bias"],
                  window=c["window"], layout=c["layout"])
    if k == "layer":
        # A step of the engine: the fog parameters are set, then every layer runs.
        KESSIE_STATE.update(fog_alpha=0.5, fog_start=0.5, prompt_len=s["meta"].max_seq_len, recall_positions=s["recall"],
                            recall_boost=0.1)
        out = [s["impl"].forward(None, q, kk, v, cache, s["meta"])
               for q, kk, v, cache in zip(s["q"], s["k"], s["v"], s["caches"])]
        return {"out": out, "caches": s["caches"]}
    if k == "dense":
        if c["fog"]:
            return s["kernels"].fused_fog_attention(s["q"], s["k"], s["v"], s["w"], window_size=c["window"],
                                                    causal=c["causal"], stream=s["stream"])
        return s["kernels"].windowed_attention(s["q"], s["k"], s["v"], window_size=c["window"], causal=c["causal"],
                                               stream=s["stream"])
    if k == "remap":
        ops.rope_remap_paged(s["pool"], s["orig"], s["tgt"], c["theta"], page_list=s["pages"], layout=c["layout"])
        return s["pool"]
    if k == "inject":
        ops.page_insert(s["pool"], s["new_k"], s["new_v"], s["pages"], s["valid"], s["positions"], 1234,
                        orig_pos=s["orig"], tgt_pos=s["tgt"], rope_theta=c["theta"], layout=c["layout"])
        return {"pool": s["pool"], "valid": s["valid"], "positions": s["positions"]}
    if k == "evict":
        valid = s["valid"].clone()  # the pass can be repeated
        evicted, _, tables, lens, idx, count = ops.page_evict_compact(s["scores"], valid, s["tables"], s["lens"])
        n, keep = c["seqs"] * c["width"], s["staging"].shape[0]
        kv = ops.page_gather(s["pool"], idx, count, out=s["staging"], n=keep)
        return {"valid": valid, "evicted": evicted[:n - keep], "tables": tables, "lens": lens, "idx": idx[:keep],
                "count": count, "kv": kv}
    sims, ids, scores = ops.index_query(s["embeds"], s["query"], top_k=c["top_k"])
    return {"sims": sims, "ids": ids, "scores": scores}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v, first, scale, window, causal, vscale=None, bias=None):
    """q [R, Hq, D] at positions first.. over k, v [N, Hkv, D], in float64: [R, Hq, D]."""
    r, hq, d = q.shape
    n, hkv = k.shape[:2]
    grp = hq // hkv
    out = torch.empty(r, hq, d, dtype=torch.float64, device=q.device)
    step = max(1, int(3e8 // (grp * n)))
    for h in range(hkv):
        kh = k[:, h].double().t().contiguous()
        vh = v[:, h].double().contiguous()
        if vscale is not None:
            vh = vh * vscale[:n, None].double()
        for r0 in range(0, r, step):
            r1 = min(r, r0 + step)
            lo = max(0, first + r0 - window + 1) if window else 0
            hi = min(n, first + r1) if causal or window else n
            qs = q[r0:r1, h * grp:(h + 1) * grp].double().reshape(-1, d)
            sc = (qs @ kh[:, lo:hi].contiguous()).view(r1 - r0, grp, hi - lo) * scale
            if bias is not None:
                sc += bias[lo:hi].double()
            dist = torch.arange(first + r0, first + r1, device=q.device)[:, None] - torch.arange(lo, hi, device=q.device)
            hide = torch.zeros_like(dist, dtype=torch.bool)
            if causal or window:
                hide |= dist < 0
            if window:
                hide |= dist >= window
            sc.masked_fill_(hide[:, None], -math.inf)
            p = torch.softmax(sc, -1).view(-1, hi - lo)
            out[r0:r1, h * grp:(h + 1) * grp] = (p @ vh[lo:hi]).view(r1 - r0, grp, d)
    return out


def _gathered(view, row, n):
    page = view.shape[1]
    return view[row[:-(-n // page)].long()].reshape(-1, view.shape[2], view.shape[3])[:n]


def _rotated(k, orig, tgt, theta):
    """K [T, H, D] moved from orig to tgt.  The angles are the operator's own (position difference times the
    fp32 frequency, in fp32); their sines, cosines and the rotation are taken in float64."""
    half = k.shape[-1] // 2
    inv = (1.0 / (theta ** (torch.arange(half, dtype=torch.float32) / half))).to(k.device)
    a = torch.outer((tgt - orig).float(), inv).double()[:, None]
    k1, k2 = k[..., :half].double(), k[..., half:].double()
    return torch.cat([k1 * a.cos() - k2 * a.sin(), k1 * a.sin() + k2 * a.cos()], -1)


def exact(case, seed):
    k = case["kind"]
    if k == "evict":
        return None  # whole numbers and copied bytes
    s = prepare(case, seed)
    scale = case["d"] ** -0.5
    if k in ("decode", "prefill"):
        kv, vv = _kv(s["pool"], case["layout"])
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        for i, (r, n) in enumerate(_seqs(case)):
            q = s["q"][i].view(r, case["hq"], case["d"])
            o = _attend(q, _gathered(kv, s["table"][i], n), _gathered(vv, s["table"][i], n), n - r, scale, case["window"],
                        True, s["vscale"], None if s["bias"] is None else s["bias"][i])
            out[i] = o.view(out[i].shape)
        return out
    if k == "layer":
        meta, outs = s["meta"], []
        for q, kk, v, cache in zip(s["q"], s["k"], s["v"], s["caches"]):
            kv, vv = _kv(cache, case["layout"])
            at, slot = meta.slot_mapping // case["page"], meta.slot_mapping % case["page"]
            kv[at, slot] = kk
            vv[at, slot] = v
            out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
            r0 = 0
            for i, (r, n) in enumerate(_seqs(case)):
                bias = _fog_bias(n, _DT[case["dtype"]])
                for p in s["recall"]:
                    if p < n:
                        bias[p] = 0.1
                out[r0:r0 + r] = _attend(q[r0:r0 + r], _gathered(kv, meta.block_table[i], n),
                                         _gathered(vv, meta.block_table[i], n), n - r, scale, case["window"], True,
                                         None, bias)
                r0 += r
            outs.append(out.view(out.shape[0], -1))
        return {"out": outs, "caches": None}
    if k == "dense":
        out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
        for b in range(case["batch"]):
            q, kk, v = (t[b].transpose(0, 1) for t in (s["q"], s["k"], s["v"]))
            out[b] = _attend(q, kk, v, 0, scale, case["window"], case["causal"],
                             s["w"] if case["fog"] else None).transpose(0, 1)
        return out
    if k in ("remap", "inject"):
        t = torch.arange(case["tokens"], device="cuda")
        at, slot = s["pages"].long()[t // case["page"]], t % case["page"]
        pool = s["pool"].double()
        kv, vv = _kv(pool, case["layout"])
        kv[at, slot] = _rotated(kv[at, slot] if k == "remap" else s["new_k"], s["orig"], s["tgt"], case["theta"])
        if k == "remap":
            return pool
        vv[at, slot] = s["new_v"].double()
        return {"pool": pool, "valid": None, "positions": None}
    e, q = s["embeds"].double(), s["query"].double()
    sims = (e @ q) / (e.norm(dim=1) * q.norm())
    return {"sims": sims, "ids": None, "scores": sims.topk(case["top_k"]).values}


def tolerance(case):
    k = case["kind"]
    if k == "evict":
        return "exact"
    if k == "index":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    if k in ("remap", "inject"):
        # One rounding of K to its type (an outlying value differs by one unit in its last place).
        return {"bf16": {"rel": 2e-3, "max": 2e-2}, "fp16": {"rel": 3e-4, "max": 2e-3}}[case["dtype"]]
    dt = "fp16" if k == "dense" else case["dtype"]
    return {"bf16": {"rel": 1e-2, "max": 0.2}, "fp16": {"rel": 1.5e-3, "max": 0.04}, "fp32": {"rel": 1e-5, "max": 2e-4}}[dt]
