"""The forms of the ping-pong prefill kernel (pa_prefill_pp.hip) that the library picks from a
launch's work-groups (W of 128 rows: q-tiles x KV heads x sequences) and its tables' width:
KSPLIT (two teams of waves on every other key tile), SOLO (one team) and SHARED, at the edges of their ranges, dense and
INT8, head_dim 64 and 128, ragged batches with an empty sequence, heads per KV head that do not
divide a q-tile. Tolerances against the double-accumulated oracle as everywhere: max abs
<= 2e-2, for INT8 plus one bf16 unit of the reference value."""
import math

import numpy as np
import pytest
import torch

import tileinfer_hip as ti
from helpers import randn, rng, smoothing
from oracle import oracle as orc
from test_prefill_pick import KSPLIT, NONE, SHARED, SOLO, pick

pytestmark = pytest.mark.gpu
BE = ti.HipBackend()

# name (its first word is the form, others take the kernels outside this one): (cache, D, heads,
# kv_heads, page_size, sequences (start, n), causal[, block-table width in positions])
CASES = {
    "paired16_ragged": ("bf16", 128, 32, 8, 16, [(700, 40), (0, 130), (0, 0)], True),   # W = 120: none
    "ksplit_dense_first": ("bf16", 128, 32, 8, 16, [(0, 520)], True),            # W = 136
    "ksplit_dense_odd_tiles": ("bf16", 128, 32, 8, 64, [(33, 700)], True),
    "ksplit_dense_non_causal": ("bf16", 128, 32, 8, 16, [(77, 641)], False),
    "ksplit_dense_g3": ("bf16", 128, 24, 8, 32, [(10, 850)], True, 2048),        # 42 positions a q-tile
    "ksplit_dense_ragged": ("bf16", 128, 32, 8, 16, [(700, 40), (0, 130), (0, 0), (900, 1), (5, 300)], True, 2048),
    "ksplit_dense_two_tiles": ("bf16", 128, 32, 8, 16, [(60 * (b % 4), 33 + b) for b in range(16)], True),
    "ksplit_dense_d64": ("bf16", 64, 32, 8, 32, [(5, 700)], True),
    "ksplit_dense_d64_non_causal": ("bf16", 64, 16, 8, 16, [(100, 650), (0, 650)], False),
    "ksplit_int8_first": ("int8", 128, 32, 8, 16, [(0, 1030)], True, 2048),      # W = 264
    "int8_ragged": ("int8", 128, 32, 8, 64, [(300, 299), (0, 31), (0, 0), (65, 300), (1, 1)], True),
    "int8_d64": ("int8", 64, 16, 8, 16, [(33, 640), (0, 600)], True),
    "solo_dense_short": ("bf16", 128, 32, 8, 16, [(17 * b, 129 + b) for b in range(16)], True),
    "solo_dense_two_tiles": ("bf16", 128, 32, 8, 16, [(3 * b, 33 + b % 8) for b in range(32)], True),
    "solo_dense_d64": ("bf16", 64, 32, 8, 64, [(0, 700), (100, 300), (0, 0), (900, 650)], True),
    "solo_dense_d64_non_causal": ("bf16", 64, 32, 8, 16, [(31, 500), (0, 320), (7, 513), (64, 33), (0, 1)], False),
    "solo_int8": ("int8", 128, 32, 8, 16, [(0, 700), (333, 650), (0, 0), (12, 32)], True),
    "solo_int8_d64": ("int8", 64, 32, 8, 32, [(0, 700), (333, 650), (1, 1), (12, 32)], True),
    "shared_dense": ("bf16", 128, 32, 8, 16, [(5, 600), (0, 601), (950, 2), (0, 0)], True),
    # an empty sequence in a step whose first position is 0: no key tile, no page to look up
    "paired16_empty_first": ("bf16", 128, 32, 8, 16, [(0, 0), (0, 130), (700, 40)], True),
    "paired16_int8_empty_first": ("int8", 128, 32, 8, 16, [(0, 0), (0, 130), (100, 40)], True),
    "ksplit_int8_ragged": ("int8", 128, 32, 8, 64, [(300, 299), (0, 231), (0, 0), (65, 300), (1, 290)], True, 2048),
    "ksplit_int8_d64": ("int8", 64, 32, 8, 16, [(33, 1040)], True, 2048),
    "shared_dense_g3": ("bf16", 128, 24, 8, 32, [(5, 700), (0, 333), (930, 85), (0, 0)], True),   # 85 positions a q-tile
}


@pytest.mark.parametrize("name", list(CASES))
def test_prefill_form(gpu, name):
    """Also with NaN in every pool row (INT8: scale) that no sequence holds, which tiles past a
    step's last key read: none may reach the output."""
    kind, D, H, KVH, P, seqs, _, width = (*CASES[name], 0)[:8]
    forms = {"shared": SHARED, "ksplit": KSPLIT, "solo": SOLO}
    assert forms.get(name.split("_")[0], NONE) == pick(
        max(n for _, n in seqs), len(seqs), max(width, P * (max(-(-(s + n) // P) for s, n in seqs) + 2)),
        sum(n for _, n in seqs), int(kind == "int8"), H, KVH, D, P)
    run_case(name, ti.TI_PATH_AUTO)


@pytest.mark.parametrize("name", ["int8_ragged", "solo_int8", "solo_int8_d64"])
def test_prefill_int8_stale_scales(gpu, name):
    """The same through the four-wave kernel, which takes the INT8 steps that no form above does."""
    run_case(name, ti.TI_PATH_PREFILL_STAGED)


def run_case(name, path):
    kind, D, H, KVH, P, seqs, causal, width = (*CASES[name], 0)[:8]
    g = rng(5200 + list(CASES).index(name))
    used = [-(-(s + n) // P) for s, n in seqs]
    pages, nmax = sum(used) + 3, max(n for _, n in seqs)
    perm = (g.permutation(pages) + 1).astype(np.int32)
    bts = np.zeros((len(seqs), max(max(used) + 2, width // P)), np.int32)
    rows = np.zeros((pages, P), bool)               # rows that hold a key
    at = 0
    for b, (s, n) in enumerate(seqs):
        bts[b, :used[b]] = perm[at:at + used[b]]
        at += used[b]
        for p in range(s + n):
            rows[bts[b, p // P] - 1, p % P] = True
    counts = [n for _, n in seqs]
    qsl = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    positions = np.concatenate([np.arange(s, s + n) for s, n in seqs]).astype(np.int32)
    q = randn(g, sum(counts), H, D, bf16=True)
    kp, vp = randn(g, pages, KVH, P, D, bf16=True), randn(g, pages, KVH, P, D, bf16=True)
    qd, scale = torch.from_numpy(q).bfloat16().cuda(), 1 / math.sqrt(D)
    stale = torch.from_numpy(~rows).cuda()[:, None].expand(pages, KVH, P)
    if kind == "int8":
        cs = smoothing(g, D)
        k, v = ti.int8_kv_pools(D, P, KVH, pages, key_smoothing=torch.from_numpy(cs))
        flat = [torch.from_numpy(np.ascontiguousarray(x.transpose(0, 2, 1, 3).reshape(-1, KVH, D))).bfloat16().cuda()
                for x in (orc.bf16_round(kp * orc.bf16_round(cs)), vp)]
        ti.store_kv_(BE, k, v, *flat, torch.arange(1, P * pages + 1, dtype=torch.int32, device="cuda"))
        pools = dict(layer_q=k.layer_q.cpu().numpy(), layer_scale=k.layer_scale.cpu().numpy(), smooth=cs)
        for half in range(2):
            k.layer_scale[half][stale] = float("nan")
    else:
        k, v = torch.from_numpy(kp).bfloat16().cuda(), torch.from_numpy(vp).bfloat16().cuda()
        pools = dict(k_pages=kp, v_pages=vp)
        k[stale] = float("nan")
        v[stale] = float("nan")
    out = torch.full_like(qd, float("nan"))
    print(f"case {name}", flush=True)
    ws = ti.attention_workspace(BE, qd, k, num_seqs=len(seqs), max_query_len=nmax, path=path)
    ti.paged_attention_(BE, out, ws, qd, k, v, torch.from_numpy(bts).cuda(), torch.from_numpy(positions).cuda(), scale,
                        causal, query_start_loc=torch.from_numpy(qsl).cuda() if len(seqs) > 1 else None, max_query_len=nmax,
                        path=path)
    got = out.float().cpu().numpy()
    for b, (s, n) in enumerate(seqs):
        if n == 0:
            continue
        ref = orc.attention(q[qsl[b]:qsl[b + 1]], bts[b], s, scale, causal, **pools)
        excess = np.abs(ref - got[qsl[b]:qsl[b + 1]]) - (2e-2 + (np.abs(ref) * 2.0 ** -8 if kind == "int8" else 0))
        assert float(np.max(excess)) <= 0, f"sequence {b}: over the tolerance by {np.max(excess)}"


# name: (cache, heads, sequences (start, n), block-table width in positions (0: just wide enough),
#        the pinned path whose kernel AUTO takes, or None: a form of the ping-pong kernel)
STAGED, PAIRED16 = ti.TI_PATH_PREFILL_STAGED, ti.TI_PATH_PREFILL_PAIRED16
ragged5 = [(831 + 300 * b, 37 + 20 * b) for b in range(5)]
PICKS = {
    # blocks of one q-tile per sequence: key splits, or the 16-row kernel where keys do not split
    "block_17_wide": ("bf16", 32, [(300, 16)] * 17, 2064, STAGED),
    "block_17_narrow": ("bf16", 32, [(300, 16)] * 17, 0, PAIRED16),
    "block_17_1040": ("bf16", 32, [(300, 16)] * 17, 1040, None),
    "block_23_wide": ("bf16", 32, [(40 * b, 16 - b % 8) for b in range(23)], 4096, STAGED),
    "block_24_wide": ("bf16", 32, [(40 * b, 16 - b % 8) for b in range(24)], 4096, None),
    "block_32": ("bf16", 32, [(40 * (b % 9), 16) for b in range(32)], 2064, PAIRED16),
    "block_63": ("bf16", 32, [(40 * (b % 9), 16) for b in range(63)], 0, PAIRED16),
    "block_64": ("bf16", 32, [(40 * (b % 9), 16) for b in range(64)], 0, None),
    "block_int8_32": ("int8", 32, [(40 * (b % 9), 16) for b in range(32)], 2064, PAIRED16),
    "block_int8_64": ("int8", 32, [(40 * (b % 9), 16) for b in range(64)], 1024, PAIRED16),
    "block_int8_64_narrow": ("int8", 32, [(40 * (b % 9), 16) for b in range(64)], 0, None),
    "block_int8_65": ("int8", 32, [(40 * (b % 9), 16) for b in range(65)], 0, None),
    # few q-tiles per sequence
    "three_tiles_narrow": ("bf16", 32, [(60, 66)] * 6, 0, PAIRED16),
    "three_tiles_1040": ("bf16", 32, [(60, 66)] * 6, 1040, None),
    "int8_20x40": ("int8", 32, [(70, 40)] * 20, 2064, PAIRED16),
    "int8_ragged": ("int8", 32, ragged5, 4096, PAIRED16),
    "int8_short_beyond_one_round": ("int8", 32, [(9, 180)] * 7, 0, STAGED),
    "short_beyond_one_round": ("bf16", 32, [(b, 123 + 10 * b) for b in range(6)], 0, STAGED),
    "short_of_nine_tiles": ("bf16", 32, [(b, 257 + 10 * b) for b in range(4)], 0, None),
    "g3_late_start": ("bf16", 24, [(0, 850)], 0, PAIRED16),
    "g3_first": ("bf16", 24, [(0, 890)], 0, None),
}


@pytest.mark.parametrize("name", list(PICKS))
def test_prefill_pick(gpu, name):
    """The kernel AUTO takes on each side of the pick's lines, by bit-equality with the pinned one
    (whose MFMA shape or order of key tiles no ping-pong form shares), and its result on the first
    and the last sequence."""
    kind, H, seqs, width, like = PICKS[name]
    D, KVH, P, B = 128, 8, 16, len(seqs)
    g = rng(5400 + list(PICKS).index(name))
    used = [-(-(s + n) // P) for s, n in seqs]
    pages, nmax = sum(used) + 1, max(n for _, n in seqs)
    bts = np.zeros((B, max(width // P, max(used))), np.int32)
    ids = iter(g.permutation(pages) + 1)
    for b in range(B):
        bts[b, :used[b]] = [next(ids) for _ in range(used[b])]
    qsl = np.concatenate([[0], np.cumsum([n for _, n in seqs])]).astype(np.int32)
    q = randn(g, qsl[-1], H, D, bf16=True)
    kp, vp = randn(g, pages, KVH, P, D, bf16=True), randn(g, pages, KVH, P, D, bf16=True)
    k, v = torch.from_numpy(kp).bfloat16().cuda(), torch.from_numpy(vp).bfloat16().cuda()
    pools = dict(k_pages=kp, v_pages=vp)
    if kind == "int8":
        flat = [x.transpose(1, 2).reshape(-1, KVH, D).contiguous() for x in (k, v)]
        k, v = ti.int8_kv_pools(D, P, KVH, pages)
        ti.store_kv_(BE, k, v, *flat, torch.arange(1, P * pages + 1, dtype=torch.int32, device="cuda"))
        pools = dict(layer_q=k.layer_q.cpu().numpy(), layer_scale=k.layer_scale.cpu().numpy(), smooth=np.ones(D, np.float32))
    qd, scale = torch.from_numpy(q).bfloat16().cuda(), 1 / math.sqrt(D)
    pos = torch.cat([torch.arange(s, s + n) for s, n in seqs]).to(torch.int32).cuda()
    outs = []
    for path in (ti.TI_PATH_AUTO, like or (PAIRED16 if kind == "int8" else STAGED)):
        print(f"pick {name} path {path}", flush=True)
        ws = ti.attention_workspace(BE, qd, k, num_seqs=B, max_query_len=nmax, path=path)
        outs.append(torch.full_like(qd, float("nan")))
        ti.paged_attention_(BE, outs[-1], ws, qd, k, v, torch.from_numpy(bts).cuda(), pos, scale,
                            query_start_loc=torch.from_numpy(qsl).cuda(), max_query_len=nmax, path=path)
    assert torch.equal(*outs) == (like is not None)
    got = outs[0].float().cpu().numpy()
    for b in (0, B - 1):
        ref = orc.attention(q[qsl[b]:qsl[b + 1]], bts[b], seqs[b][0], scale, True, **pools)
        excess = np.abs(ref - got[qsl[b]:qsl[b + 1]]) - (2e-2 + (np.abs(ref) * 2.0 ** -8 if kind == "int8" else 0))
        assert float(np.max(excess)) <= 0, f"sequence {b}: over the tolerance by {np.max(excess)}"


@pytest.mark.parametrize("D,seqs,n,start,like", [(128, 1, 600, 0, PAIRED16), (128, 5, 128, 100, PAIRED16),
                                                 (128, 20, 16, 1008, STAGED), (64, 3, 240, 100, STAGED),
                                                 (64, 64, 16, 100, STAGED)])
def test_prefill_form_rounds_no_more(gpu, D, seqs, n, start, like):
    """The error against 64 bits (2-norm, three seeds) is no larger than that of the kernel that takes
    such a step otherwise: 0.5 % for the seeds. Without the first steps' eager rescale it was 1.4 to
    6 % larger, with it 0.3 to 1.6 % smaller."""
    H, KVH, P = 32, 8, 16
    per = -(-(start + n) // P)
    assert pick(n, seqs, P * per, heads=H, kv_heads=KVH, D=D) != NONE
    norms = np.zeros(2)
    for seed in range(3):
        g = rng(5500 + seed + n + D)
        bts = (g.permutation(seqs * per) + 1).astype(np.int32).reshape(seqs, per)
        q, kp = randn(g, seqs * n, H, D, bf16=True), randn(g, seqs * per, KVH, P, D, bf16=True)
        vp = randn(g, seqs * per, KVH, P, D, bf16=True)
        ref = np.concatenate([orc.attention(q[b * n:(b + 1) * n], bts[b], start, 1 / math.sqrt(D), True, kp, vp)
                              for b in range(seqs)])
        qd, k, v = (torch.from_numpy(x).bfloat16().cuda() for x in (q, kp, vp))
        pos = torch.arange(start, start + n, dtype=torch.int32, device="cuda").repeat(seqs)
        for i, path in enumerate((ti.TI_PATH_AUTO, like)):
            out = torch.empty_like(qd)
            ws = ti.attention_workspace(BE, qd, k, num_seqs=seqs, max_query_len=n, path=path)
            ti.paged_attention_(BE, out, ws, qd, k, v, torch.from_numpy(bts).cuda(), pos, 1 / math.sqrt(D), max_query_len=n,
                                path=path)
            norms[i] += np.linalg.norm(out.float().cpu().numpy() - ref)
    assert norms[0] <= 1.005 * norms[1], norms[0] / norms[1]
