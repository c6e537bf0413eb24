"""Performance cases: attention blocks of a model step over the paged KV cache.

Every case is what a runner does between a layer's qkv projection and its output
projection: `attention_inputs_` (optional q/k RMSNorm, RoPE, queries out, keys and values
into the cache pages) and then `paged_attention_` over the cached and the new positions.
Cases differ in the shape of the step (one token per sequence, a drafted block, a prompt, a
chunk on a cached prefix), the batch and its lengths, the heads, the page size, the cache
type and whether the step is a captured graph over several layers (as a runner captures its
decode steps) or eager calls.
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "tileinfer.jl_amd"))

import tileinfer_hip as ti  # noqa: E402

BE = ti.HipBackend()
THETA, EPS = 1e6, 1e-6
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, **kw):
    # ctx / new: cached and new positions per sequence, drawn between the bounds from `lens`
    c = dict(name=name, dtype="bf16", kv="dense", heads=32, kv_heads=8, head_dim=128, page=64, seqs=1, ctx_min=0, ctx=0,
             new_min=1, new=1, causal=True, norm=True, layers=1, graph=False, lens=1)
    c.update(kw)
    return c


def listed():
    return [
        # one token of a small float32 model, eager: the smallest call, all latency
        _case("token_fp32", dtype="fp32", heads=16, page=16, ctx_min=1023, ctx=1023),
        # one chat: the attention of 16 layers of a one-token step, captured
        _case("token_graph", ctx_min=3000, ctx=3000, layers=16, graph=True),
        # a few chats of very different lengths, one token each, captured
        _case("decode_ragged_b8", page=16, seqs=8, ctx_min=1023, ctx=8191, layers=8, graph=True),
        # a serving batch of one-token steps, eager: the benchmark's shape
        _case("decode_b32", page=16, seqs=32, ctx_min=4095, ctx=4095, norm=False),
        # many short chats on a model with 64-wide heads, captured
        _case("decode_short_b100_d64", head_dim=64, seqs=100, ctx_min=20, ctx=1000, norm=False, layers=8, graph=True),
        # long contexts on an INT8 cache
        _case("decode_int8_32k", kv="int8", page=16, seqs=8, ctx_min=32767, ctx=32767, norm=False),
        # speculative decoding: a drafted block of 16 tokens per sequence is verified
        _case("verify_b16", page=16, seqs=16, ctx_min=4096, ctx=4096, new_min=16, new=16),
        # a prompt from scratch
        _case("prefill_512", page=16, new_min=512, new=512),
        # a prompt whose first 1024 tokens are already cached
        _case("chunk_512_on_1024", page=16, ctx_min=1024, ctx=1024, new_min=512, new=512),
        # a batch of prompts of mixed lengths, 64-wide heads
        _case("prompts_b8_d64", head_dim=64, seqs=8, new_min=100, new=2000, norm=False),
        # a chunk of a long document on an INT8 cache
        _case("chunk_int8_1500_on_3000", kv="int8", ctx_min=3000, ctx=3000, new_min=1500, new=1500),
        # a long document in one prompt: the largest call
        _case("prefill_8192", new_min=8192, new=8192),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / (3 if case["dtype"] == "fp32" else 50))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        step = rng.choice(["token", "token", "block", "prompt", "prompt", "chunk"])
        dtype, kv = rng.choice([("bf16", "dense")] * 6 + [("bf16", "int8")] * 3 + [("fp32", "dense")])
        heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 8), (24, 8), (32, 4), (64, 8)])
        c = dict(dtype=dtype, kv=kv, heads=heads, kv_heads=kv_heads, head_dim=rng.choice([128, 128, 128, 64]),
                 page=rng.choice([16, 64, 64, 32]), causal=True, norm=rng.random() < 0.5, layers=1, graph=False,
                 lens=rng.randrange(1 << 30))
        ragged = rng.random() < 0.6
        if step == "token":
            c["seqs"], c["ctx"], c["new"] = _log(rng, 1, 128), _log(rng, 16, 32768), 1
            c["ctx_min"] = rng.randint(c["ctx"] // 8, c["ctx"]) if ragged else c["ctx"]
            c["graph"] = rng.random() < 0.6
            c["layers"] = rng.randint(2, 16) if c["graph"] else 1
        elif step == "block":
            c["seqs"], c["ctx"], c["new"] = _log(rng, 1, 32), _log(rng, 64, 8192), rng.randint(2, 16)
            c["ctx_min"] = rng.randint(c["ctx"] // 8, c["ctx"]) if ragged else c["ctx"]
            c["causal"] = rng.random() < 0.7       # a drafter's own block is not causal
        else:
            c["seqs"] = rng.choice([1, 1, 1, rng.randint(2, 16)])
            c["new"] = _log(rng, 17, 8192)
            c["ctx"] = _log(rng, 16, 8192) if step == "chunk" else 0
            c["ctx_min"] = rng.randint(c["ctx"] // 8, c["ctx"]) if ragged else c["ctx"]
        several = step in ("prompt", "chunk") and ragged and c["seqs"] > 1
        c["new_min"] = rng.randint(max(1, c["new"] // 16), c["new"]) if several else c["new"]
        if _cost(c) <= most and sum(_pages(c)) * c["layers"] * c["page"] * c["kv_heads"] * c["head_dim"] < 1 << 30:
            return c


def _lengths(case):
    """Cached and new positions of each sequence."""
    r = random.Random(case["lens"])
    return [(r.randint(case["ctx_min"], case["ctx"]), r.randint(case["new_min"], case["new"])) for _ in range(case["seqs"])]


def _pages(case):
    return [-(-(c + n) // case["page"]) for c, n in _lengths(case)]


def _inputs(case, seed):
    """What the seed draws: per layer the qkv rows, the norm weights, and the cache pages as
    they are before the step; block tables, positions and slots of the new tokens."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    T, P, D, Hk, Hq, L = DTYPES[case["dtype"]], case["page"], case["head_dim"], case["kv_heads"], case["heads"], case["layers"]
    lens, per = _lengths(case), _pages(case)
    used = sum(per)
    pages, n = used + 3, sum(x for _, x in lens)
    # tables as wide as the next power of two of positions, as a runner grows them
    width = (1 << (max(c + x for c, x in lens) - 1).bit_length()) // P + 1
    ids = (torch.randperm(pages, generator=g, device="cuda")[:used] + 1).to(torch.int32)
    tables = torch.zeros((len(lens), width), dtype=torch.int32, device="cuda")
    positions, slots, at = [], [], 0
    for b, (c, x) in enumerate(lens):
        tables[b, :per[b]] = ids[at:at + per[b]]
        at += per[b]
        p = torch.arange(c, c + x, device="cuda")
        positions.append(p)
        slots.append((tables[b, p // P].long() - 1) * P + p % P + 1)
    s = dict(tables=tables, positions=torch.cat(positions).to(torch.int32), slots=torch.cat(slots).to(torch.int32))
    starts = torch.tensor([0] + [x for _, x in lens]).cumsum(0)
    s["query_start"] = None if case["new_min"] == case["new"] else starts.to(torch.int32).cuda()
    s["rows"] = starts.tolist()
    s["qkv"] = torch.randn((L, n, (Hq + 2 * Hk) * D), generator=g, device="cuda").to(T)
    if case["norm"]:
        s["norms"] = (torch.rand((L, 2, D), generator=g, device="cuda") + 0.5).to(T)
    if case["kv"] == "dense":
        s["k"] = torch.randn((L, pages, Hk, P, D), generator=g, device="cuda").to(T)
        s["v"] = torch.randn((L, pages, Hk, P, D), generator=g, device="cuda").to(T)
    else:
        s["kv_q"], s["kv_scale"] = [], []
        for _ in range(L):
            q = torch.empty((2, pages, Hk, P, D), dtype=torch.int8, device="cuda")
            scale = torch.empty((2, pages, Hk, P), device="cuda")
            for half in range(2):
                for i in range(0, pages, 4096):
                    x = torch.randn(q[half, i:i + 4096].shape, generator=g, device="cuda")
                    top = x.abs().amax(-1, keepdim=True)
                    q[half, i:i + 4096] = torch.floor(x * (127 / top) + 0.5).to(torch.int8)
                    scale[half, i:i + 4096] = (top / 127)[..., 0]
            s["kv_q"].append(q)
            s["kv_scale"].append(scale)
    return s


def _cos_sin(case):
    top = max(c + n for c, n in _lengths(case))
    D = case["head_dim"]
    inv = THETA ** (-torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
    a = torch.arange(top, dtype=torch.float64, device="cuda")[:, None] * torch.cat([inv, inv])[None]
    return a.cos(), a.sin()


def prepare(case, seed):
    s = _inputs(case, seed)
    T, D = DTYPES[case["dtype"]], case["head_dim"]
    L, n, Hq = case["layers"], s["qkv"].shape[1], case["heads"]
    s["table"] = ti.RotaryTable.from_arrays(*_cos_sin(case), T)
    s["q"] = torch.zeros((L, n, Hq, D), dtype=T, device="cuda")
    s["out"] = torch.zeros_like(s["q"])
    s["scale"], s["causal"], s["seqs"], s["new"] = 1 / math.sqrt(D), case["causal"], case["seqs"], case["new"]
    if case["kv"] == "dense":
        s["pools"] = [(s["k"][i], s["v"][i]) for i in range(L)]
    else:
        s["pools"] = []
        for i, (kv_q, kv_scale) in enumerate(zip(s["kv_q"], s["kv_scale"])):
            smooth = ti.key_smoothing(s["norms"][i, 1]) if case["norm"] else None
            pair = ti.int8_kv_pools(D, case["page"], case["kv_heads"], kv_q.shape[1], smooth)
            pair[0].layer_q.copy_(kv_q)
            pair[0].layer_scale.copy_(kv_scale)
            s["pools"].append(pair)
        del s["kv_q"], s["kv_scale"]
    s["workspace"] = ti.attention_workspace(BE, s["q"][0], s["pools"][0][0], num_seqs=s["seqs"], max_query_len=s["new"])
    s["views"] = [(s["q"][i], s["out"][i], s["qkv"][i]) + ((s["norms"][i, 0], s["norms"][i, 1]) if case["norm"] else (None, None))
                  for i in range(L)]
    s["graph"] = None
    if case["graph"]:
        _step(s)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _step(s)
    return s


def _step(s):
    for (k, v), (q, out, qkv, q_norm, k_norm) in zip(s["pools"], s["views"]):
        ti.attention_inputs_(BE, q, k, v, qkv, q_norm, k_norm, s["table"], s["positions"], s["slots"], EPS)
        ti.paged_attention_(BE, out, s["workspace"], q, k, v, s["tables"], s["positions"], s["scale"], s["causal"],
                            query_start_loc=s["query_start"], max_query_len=s["new"])


def run(s):
    if s["graph"] is not None:
        s["graph"].replay()
    else:
        _step(s)
    if "k" in s:
        return {"q": s["q"], "out": s["out"], "k": s["k"], "v": s["v"]}
    return {"q": s["q"], "out": s["out"], "kv": [(k.layer_q, k.layer_scale) for k, _ in s["pools"]]}


def work(case):
    D, Hk, Hq, L = case["head_dim"], case["kv_heads"], case["heads"], case["layers"]
    e = 2 if case["dtype"] == "bf16" else 4
    row = D * e if case["kv"] == "dense" else D + 4        # one cached key or value of one head
    moved = flops = 0
    for c, n in _lengths(case):
        # qkv and rotary rows in; queries and the result out; cached rows in, new rows out
        moved += n * ((Hq + 2 * Hk) * D * e + 2 * D * e) + 2 * n * Hq * D * e + 2 * (c + n) * Hk * row
        visible = n * c + (n * (n + 1) // 2 if case["causal"] else n * n)
        flops += 4 * D * Hq * visible
    return {"bytes": moved * L, "flops": flops * L}


def tolerance(case):
    # float32: sums of up to 8192 products in another order. bf16: probabilities and results
    # are rounded to 8 bits (measured 0.002-0.005 against 64 bits); INT8: the queries times the
    # keys' smoothing and the probabilities times the values' scales too (0.003-0.008). INT8
    # pages are written exactly, whatever computes the attention.
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 2e-4}
    return {"rel": 1e-2, "max": 0.2} if case["kv"] == "dense" else {"rel": 2e-2, "max": 0.4}


def exact(case, seed):
    s = _inputs(case, seed)
    lens, P, D, Hk, Hq = _lengths(case), case["page"], case["head_dim"], case["kv_heads"], case["heads"]
    G, f64 = Hq // Hk, torch.float64
    T = DTYPES[case["dtype"]]
    cos, sin = (x.to(T).to(f64)[s["positions"].long()][:, None] for x in _cos_sin(case))
    sign = torch.cat([-torch.ones(D // 2), torch.ones(D // 2)]).to("cuda", f64)
    page, off = (s["slots"].long() - 1) // P, (s["slots"].long() - 1) % P
    got = {"q": [], "out": []}
    got.update({"k": [], "v": []} if case["kv"] == "dense" else {"kv": []})
    for i in range(case["layers"]):
        x = s["qkv"][i].to(f64).view(-1, Hq + 2 * Hk, D)
        heads, v = x[:, :Hq + Hk], x[:, Hq + Hk:]
        if case["norm"]:
            w = s["norms"][i].to(f64)
            heads = heads / (heads.square().mean(-1, keepdim=True) + EPS).sqrt()
            heads = torch.cat([heads[:, :Hq] * w[0], heads[:, Hq:] * w[1]], 1)
        heads = heads * cos + heads.roll(D // 2, -1) * sign * sin
        q, k = heads[:, :Hq], heads[:, Hq:]
        if case["kv"] == "dense":
            for key, new in (("k", k), ("v", v)):
                pool = s[key][i].to(f64)
                pool[page, :, off] = new
                got[key].append(pool)
            pools = got["k"][-1], got["v"][-1]
            rows = [lambda ids, h, p=p: p[ids, h].reshape(-1, D) for p in pools]
        else:
            smooth = torch.ones(D, dtype=f64, device="cuda")
            if case["norm"]:
                w = w[1].abs()
                smooth = torch.maximum(w[:D // 2], w[D // 2:]).repeat(2)
            values, scales = s["kv_q"][i], s["kv_scale"][i].to(f64)
            for half, new in ((0, k / smooth), (1, v)):
                top = new.abs().amax(-1, keepdim=True)
                values[half][page, :, off] = torch.floor(new * (127 / top) + 0.5).to(torch.int8)
                scales[half][page, :, off] = (top / 127)[..., 0]
            got["kv"].append((None, scales))
            rows = [lambda ids, h, j=j, m=m: (values[j][ids, h].to(f64) * scales[j][ids, h][..., None]).reshape(-1, D) * m
                    for j, m in ((0, smooth), (1, 1.0))]
        out = torch.empty_like(q)
        for b, (c, n) in enumerate(lens):
            ids = s["tables"][b, :-(-(c + n) // P)].long() - 1
            t0 = s["rows"][b]
            for h in range(Hk):
                kk, vv = (r(ids, h)[:c + n] for r in rows)
                for t in range(0, n, 1024):
                    qq = q[t0 + t:t0 + min(n, t + 1024), h * G:(h + 1) * G]
                    m = qq.shape[0]
                    sc = (qq.reshape(-1, D) @ kk.T).view(m, G, -1) / math.sqrt(D)
                    if case["causal"]:
                        seen = torch.arange(c + n, device="cuda")[None] <= torch.arange(c + t, c + t + m, device="cuda")[:, None]
                        sc.masked_fill_(~seen[:, None], -math.inf)
                    out[t0 + t:t0 + t + m, h * G:(h + 1) * G] = (sc.softmax(-1).view(m * G, -1) @ vv).view(m, G, D)
        got["q"].append(q)
        got["out"].append(out)
    for key in set(got) - {"kv"}:
        got[key] = torch.stack(got[key])
    return got
