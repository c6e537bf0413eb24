"""The native call path of the Python op interface (csrc/py_calls.cpp) against backend.py's own
checks and ctypes calls: the same results for every form it takes, the same errors for what
it leaves to them."""
import math

import numpy as np
import pytest
import torch

import tileinfer_hip as ti
from helpers import rng
from tileinfer_hip import _lib

pytestmark = pytest.mark.gpu
BE = ti.HipBackend()


class _NotPlain:
    """A native path that leaves every call to backend.py."""
    def __getattr__(self, name):
        return lambda *a: -1


class _Counted:
    def __init__(self, calls):
        self.calls, self.made = calls, 0

    def __getattr__(self, name):
        def f(*a):
            status = getattr(self.calls, name)(*a)
            self.made += status == 0
            return status
        return f


def _step(dtype, int8, B, n, one):
    """One step through every op; returns its outputs."""
    g = torch.Generator(device="cuda").manual_seed(7 + B + n)
    D, Hq, Hk, P, L = 128, 16, 8, 16, 70
    per = (L + n) // P + 1
    pages = B * per + 1
    rand = lambda *s: torch.randn(s, generator=g, device="cuda").to(dtype)  # noqa: E731
    bts = (torch.randperm(pages, generator=g, device="cuda")[:B * per] + 1).to(torch.int32).view(B, per)
    pos = torch.arange(L, L + n, device="cuda", dtype=torch.int32).repeat(B)
    slots = torch.cat([(bts[b][(pos[:n] // P).long()] - 1) * P + pos[:n] % P + 1 for b in range(B)]).to(torch.int32)
    table = ti.RotaryTable.build(D, 128, 1e6, dtype)
    if int8:
        k, v = ti.int8_kv_pools(D, P, Hk, pages, ti.key_smoothing(rand(D)))
    else:
        k, v = rand(pages, Hk, P, D), rand(pages, Hk, P, D)
    x, kk, vv = rand(B * n, Hq, D), rand(B * n, Hk, D), rand(B * n, Hk, D)
    w = rand(D)
    ti.store_kv_(BE, k, v, kk, vv, slots)
    q = ti.rope(BE, ti.rmsnorm(BE, x, w, 1e-6), table.cos, table.sin, pos)
    q2 = torch.empty_like(q)
    ti.attention_inputs_(BE, q2, k, v, rand(B * n, (Hq + 2 * Hk) * D), w if n > 1 else None, w if n > 1 else None, table,
                         pos, slots, 1e-6)
    outs = [q, q2] + ([k.layer_q, k.layer_scale] if int8 else [k, v])
    qsl = torch.arange(0, B * n + 1, n, dtype=torch.int32, device="cuda")
    for kw in ({}, {"query_start_loc": qsl, "max_query_len": n}, {"max_query_len": n, "causal": False}):
        out = torch.empty_like(q)
        ws = ti.attention_workspace(BE, q, k, num_seqs=B, max_query_len=n)
        ti.paged_attention_(BE, out, ws, q, k, v, bts, pos, 1 / math.sqrt(D), **kw)
        outs.append(out)
    if one:
        outs.append(ti.attention(BE, q, k, v, bts[0], pos, 0.1))
        outs.append(ti.attention(BE, q, k, v, bts, pos, 1, causal=False))   # a [1][width] table, an int scale
    return outs


@pytest.mark.parametrize("dtype,int8,B,n", [(torch.bfloat16, False, 1, 1), (torch.bfloat16, True, 3, 1),
                                            (torch.bfloat16, False, 2, 40), (torch.float32, False, 1, 5),
                                            (torch.bfloat16, True, 1, 33)])
def test_native_calls_match(gpu, monkeypatch, dtype, int8, B, n):
    counted = _Counted(_lib.native())
    monkeypatch.setattr(_lib, "calls", counted)
    got = _step(dtype, int8, B, n, B == 1)
    assert counted.made == 7 + 2 * (B == 1)          # every call was a plain one
    monkeypatch.setattr(_lib, "calls", _NotPlain())
    want = _step(dtype, int8, B, n, B == 1)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_native_calls_leave_the_rest(gpu):
    """Forms that only backend.py takes still work; what it refuses is refused alike."""
    g = rng(1)
    D, H, P = 128, 8, 16
    mk = lambda *s, t=torch.bfloat16: torch.from_numpy(g.standard_normal(s, dtype=np.float32)).to(t).cuda()  # noqa: E731
    q, k, v = mk(2, H, D), mk(4, H, P, D), mk(4, H, P, D)
    bt, pos = torch.tensor([3, 1, 0], dtype=torch.int32).cuda(), torch.tensor([5, 6], dtype=torch.int32).cuda()
    ws = ti.attention_workspace(BE, q, k)
    want = ti.attention(BE, q, k, v, bt, pos, 0.25)

    def run(**kw):
        a = dict(out=torch.empty_like(q), ws=ws, q=q, k=k, v=v, bt=bt, pos=pos, scale=0.25, causal=True)
        a.update(kw)
        return ti.attention_(BE, a["out"], a["ws"], a["q"], a["k"], a["v"], a["bt"], a["pos"], a["scale"], a["causal"])

    for kw in (dict(scale=np.float64(0.25)), dict(causal=1), dict(q=torch.nn.Parameter(q)), dict(bt=bt.view(1, -1))):
        assert torch.equal(run(**kw), want)
    for kw in (dict(q=q.transpose(0, 1)), dict(pos=pos.long()), dict(pos=pos[:1]), dict(bt=bt.float()), dict(k=k.float()),
               dict(v=v[:2]), dict(out=torch.empty_like(q).float()), dict(q=q.cpu()), dict(q=q.half()), dict(scale=-1.0),
               dict(scale=float("nan")), dict(k=k[..., :64].contiguous(), v=v[..., :64].contiguous())):
        with pytest.raises(ti.ArgumentError):
            run(**kw)
    with pytest.raises(ti.WorkspaceError):
        run(ws=None, q=q[:1], out=torch.empty_like(q[:1]), pos=pos[:1])
