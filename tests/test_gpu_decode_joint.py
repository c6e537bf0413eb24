"""INT8 decode whose whole steps of three 16-key tiles share one softmax (launches of at most 256
work-groups, head_dim 128, up to 16 packed rows): key counts around whole and partial steps of
a split, several query tokens, pages of less than a tile, against the oracle over the
dequantized cache. Tolerance: max abs <= 2e-2 plus one bf16 unit of the reference value; where all
keys weigh alike, relative."""
import math

import numpy as np
import pytest
import torch

import tileinfer_hip as ti
from helpers import block_table, randn, rng, smoothing
from oracle import oracle as orc

BE = ti.HipBackend()

# (heads, kv_heads, page_size, start, n, causal); one KV head splits its keys 16 ways, 32 eight
CASES = [(4, 1, 16, 47, 1, True), (4, 1, 16, 768, 1, True), (4, 1, 16, 3071, 1, True), (4, 1, 16, 3072, 1, True),
         (4, 1, 64, 9300, 1, True), (16, 1, 16, 2400, 1, True), (4, 1, 16, 3060, 4, True), (4, 1, 16, 3060, 4, False),
         (64, 32, 16, 1000, 1, True), (64, 32, 16, 1151, 5, True), (8, 2, 4, 2303, 1, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_decode_int8_joint(gpu, case):
    H, KVH, P, start, n, causal = case
    D, L = 128, start + n
    g = rng(6100 + start + n + H)
    pages = -(-L // P) + 2
    bt = block_table(g, L, P, pages)
    q = randn(g, n, H, D, bf16=True)
    # a few keys far above the rest, so that the running max moves inside and between steps
    kp, vp = randn(g, pages, KVH, P, D, bf16=True), randn(g, pages, KVH, P, D, bf16=True)
    kp[:: max(1, pages // 7)] = orc.bf16_round(kp[:: max(1, pages // 7)] * np.float32(3))
    cs = smoothing(g, D)
    k, v = ti.int8_kv_pools(D, P, KVH, pages, key_smoothing=torch.from_numpy(cs))
    flat = [torch.from_numpy(np.ascontiguousarray(x.transpose(0, 2, 1, 3).reshape(-1, KVH, D))).bfloat16().cuda()
            for x in (orc.bf16_round(kp * orc.bf16_round(cs)), vp)]
    ti.store_kv_(BE, k, v, *flat, torch.arange(1, P * pages + 1, dtype=torch.int32, device="cuda"))
    ref = orc.attention(q, bt, start, 1 / math.sqrt(D), causal, layer_q=k.layer_q.cpu().numpy(),
                        layer_scale=k.layer_scale.cpu().numpy(), smooth=cs)
    qd = torch.from_numpy(q).bfloat16().cuda()
    out = torch.full_like(qd, float("nan"))
    print(f"case {case}", flush=True)
    ti.attention_(BE, out, ti.attention_workspace(BE, qd, k, path=ti.TI_PATH_DECODE), qd, k, v, torch.from_numpy(bt).cuda(),
                  torch.arange(start, L, dtype=torch.int32, device="cuda"), 1 / math.sqrt(D), causal, path=ti.TI_PATH_DECODE)
    excess = np.abs(ref - out.float().cpu().numpy()) - (2e-2 + np.abs(ref) * 2.0 ** -8)
    assert float(np.max(excess)) <= 0, f"over the tolerance by {np.max(excess)}"


def _marked_values(pattern, L, h):
    """Dim and size of the one value that key position p of KV head h holds: by key, or by 16-key
    tile (sizes grow with every 128 tiles, so no two tiles of one dim are alike)."""
    p = np.arange(L)
    if pattern == "key":
        return (p + 7 * h) % 128, np.ones(L, np.float32)
    return (p // 16 + 7 * h) % 128, (1 + 0.25 * (p // 16 // 128)).astype(np.float32)


def _marked_bound(ref):
    """One bf16 rounding (2^-9), doubled for the fp16 probabilities and the merge, plus 2^-9 of the
    row's RMS for dims that no key marks (the biased values' sum, 1152 N, cancels in fp32)."""
    return 2.0 ** -8 * np.abs(ref) + 2.0 ** -9 * np.sqrt(np.mean(np.square(ref), -1, keepdims=True))


@pytest.mark.parametrize("pattern,units", [("tile", (16, 48)), ("key", (1, 16, 48))])
def test_marked_values_show_every_key(pattern, units):
    """No key, tile or joint step of a case can be left out or counted twice within the bound."""
    for L in sorted({start + n for _, _, _, start, n, _ in CASES}):
        dim, size = _marked_values(pattern, L, 0)
        v = np.zeros((L, 128))
        v[np.arange(L), dim] = size
        total, ref = v.sum(0), v.mean(0)
        for unit in (u for u in units if u < L):     # (all keys twice change nothing)
            for a in range(0, L, unit):
                part, n = v[a:a + unit].sum(0), min(unit, L - a)
                for got in ((total + part) / (L + n), (total - part) / (L - n)):
                    assert (np.abs(got - ref) > _marked_bound(ref)).any(), (L, unit, a)


@pytest.mark.gpu
@pytest.mark.parametrize("pattern", ["tile", "key"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_decode_int8_joint_every_key(gpu, case, pattern):
    """Zero queries weigh all visible keys alike and every key (or tile) marks one dim, so that a
    skipped or doubled one shows (test_marked_values_show_every_key)."""
    H, KVH, P, start, n, causal = case
    D, L = 128, start + n
    g = rng(6300 + start + n + H)
    pages = -(-L // P) + 2
    bt = block_table(g, L, P, pages)
    kp, vp = randn(g, pages, KVH, P, D, bf16=True), randn(g, pages, KVH, P, D, bf16=True) * 8
    pos = np.arange(L)
    vp[bt[pos // P] - 1, :, pos % P] = 0
    for h in range(KVH):
        dim, size = _marked_values(pattern, L, h)
        vp[bt[pos // P] - 1, h, pos % P, dim] = size
    k, v = ti.int8_kv_pools(D, P, KVH, pages)
    flat = [torch.from_numpy(np.ascontiguousarray(x.transpose(0, 2, 1, 3).reshape(-1, KVH, D))).bfloat16().cuda()
            for x in (kp, vp)]
    ti.store_kv_(BE, k, v, *flat, torch.arange(1, P * pages + 1, dtype=torch.int32, device="cuda"))
    q = np.zeros((n, H, D), np.float32)
    ref = orc.attention(q, bt, start, 1 / math.sqrt(D), causal, layer_q=k.layer_q.cpu().numpy(),
                        layer_scale=k.layer_scale.cpu().numpy(), smooth=np.ones(D, np.float32))
    qd = torch.from_numpy(q).bfloat16().cuda()
    out = torch.full_like(qd, float("nan"))
    print(f"case {case} {pattern}", flush=True)
    ti.attention_(BE, out, ti.attention_workspace(BE, qd, k, path=ti.TI_PATH_DECODE), qd, k, v, torch.from_numpy(bt).cuda(),
                  torch.arange(start, L, dtype=torch.int32, device="cuda"), 1 / math.sqrt(D), causal, path=ti.TI_PATH_DECODE)
    excess = np.abs(ref - out.float().cpu().numpy()) - _marked_bound(ref)
    assert float(np.max(excess)) <= 0, f"over the tolerance by {np.max(excess)}"
