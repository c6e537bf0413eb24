"""Which form of the ping-pong prefill kernel the library picks (ti_pick_prefill_pp: host shapes
only, so no GPU), on each side of its lines. tests/test_gpu_prefill_forms.py runs the forms."""
import ctypes

import pytest

import tileinfer_hip as ti
from tileinfer_hip import _lib

NONE, SHARED, KSPLIT, SOLO = range(4)


def pick(n, seqs, keys, total=None, kind=0, heads=32, kv_heads=8, D=128, page=16):
    f = getattr(ti.load_library(), "_Z18ti_pick_prefill_ppPK17ti_attention_argsPK11ti_kv_cacheib")
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_bool]
    c = _lib.KVCache()
    c.kind, c.head_dim, c.page_size, c.kv_heads, c.num_pages = kind, D, page, kv_heads, 100
    a = _lib.AttentionArgs()
    a.dtype, a.q_heads, a.num_seqs, a.max_query_len = _lib.TI_BF16, heads, seqs, n
    a.total_tokens, a.block_table_stride = seqs * n if total is None else total, keys // page
    a.scale, a.causal = 1.0, 1
    return f(ctypes.byref(a), ctypes.byref(c), _lib.TI_PATH_AUTO, True)


@pytest.mark.parametrize("want,kw", [
    # dense head_dim 128 batches of more than 512 work-groups of 128 rows: SOLO where 256-row tiles
    # have few steps or hold little, SHARED otherwise
    (SOLO, dict(n=300, seqs=16, keys=576)),
    (SOLO, dict(n=512, seqs=16, keys=576)),
    (SOLO, dict(n=768, seqs=8, keys=1280)),
    (SHARED, dict(n=769, seqs=8, keys=1280)),
    (SHARED, dict(n=768, seqs=8, keys=1296)),
    (SHARED, dict(n=768, seqs=7, keys=1280)),
    (SHARED, dict(n=512, seqs=16, keys=8208)),
    (SHARED, dict(n=2048, seqs=8, keys=2112)),
    (SHARED, dict(n=4096, seqs=8, keys=4160)),
    (SHARED, dict(n=4096, seqs=8, keys=4160, total=8200)),
    (SOLO, dict(n=4096, seqs=8, keys=4160, total=8100)),
    (SOLO, dict(n=2000, seqs=17, keys=4112, total=2016)),
    (SHARED, dict(n=8192, seqs=1, keys=8256)),
    (SOLO, dict(n=8192, seqs=1, keys=8256, D=64)),
    (SOLO, dict(n=8192, seqs=1, keys=8256, kind=1)),
    (SHARED, dict(n=700, seqs=4, keys=1040, heads=24)),
])
def test_pick_of_large_launches(want, kw):
    assert pick(**kw) == want


@pytest.mark.parametrize("want,kw", [
    # fewer than 256 64-row q-tiles: the four-wave plan (key splits from 32 tiles of table)
    (NONE, dict(n=16, seqs=17, keys=992)),
    (KSPLIT, dict(n=16, seqs=17, keys=1008)),
    (KSPLIT, dict(n=16, seqs=17, keys=1280)),
    (NONE, dict(n=16, seqs=17, keys=1296)),
    (NONE, dict(n=16, seqs=23, keys=4112)),
    (KSPLIT, dict(n=16, seqs=24, keys=4112)),
    (NONE, dict(n=66, seqs=6, keys=4112)),
    # one q-tile of up to 64 rows
    (NONE, dict(n=16, seqs=32, keys=4112)),
    (NONE, dict(n=16, seqs=63, keys=4112)),
    (SOLO, dict(n=16, seqs=64, keys=4112)),
    (KSPLIT, dict(n=17, seqs=32, keys=4112)),
    (KSPLIT, dict(n=32, seqs=48, keys=48)),
    (NONE, dict(n=32, seqs=48, keys=48, kind=1)),
    (KSPLIT, dict(n=32, seqs=48, keys=4112, kind=1)),
    (NONE, dict(n=16, seqs=64, keys=4112, kind=1)),
    (SOLO, dict(n=16, seqs=65, keys=4112, kind=1)),
    (SOLO, dict(n=16, seqs=64, keys=992, kind=1)),
    (SOLO, dict(n=16, seqs=64, keys=4112, kind=1, D=64)),
    (NONE, dict(n=16, seqs=63, keys=992, kind=1)),
    (SOLO, dict(n=92, seqs=24, keys=144, kind=1, total=1476)),
    # INT8: the 16-row kernel's range, tokens held
    (NONE, dict(n=40, seqs=20, keys=2064, kind=1)),
    (NONE, dict(n=119, seqs=5, keys=4112, kind=1, total=357)),
    (KSPLIT, dict(n=121, seqs=5, keys=144, kind=1)),
    (NONE, dict(n=121, seqs=5, keys=1008, kind=1)),
    (NONE, dict(n=121, seqs=5, keys=144, kind=1, total=604)),
    (NONE, dict(n=128, seqs=8, keys=144, kind=1)),
    (NONE, dict(n=600, seqs=1, keys=608, kind=1)),
    (NONE, dict(n=1024, seqs=1, keys=4112, kind=1)),
    (KSPLIT, dict(n=1025, seqs=1, keys=4112, kind=1)),
    (KSPLIT, dict(n=1184, seqs=2, keys=4112, kind=1, total=1723)),
    (NONE, dict(n=1184, seqs=2, keys=4112, kind=1, total=1723, D=64)),
    (SOLO, dict(n=1184, seqs=2, keys=4112, kind=1)),
    (NONE, dict(n=534, seqs=2, keys=1040, kind=1)),
    (NONE, dict(n=534, seqs=2, keys=1280, kind=1)),
    (KSPLIT, dict(n=534, seqs=2, keys=1296, kind=1)),
    # one round and more, with few key tiles and many
    (NONE, dict(n=512, seqs=1, keys=1040)),
    (KSPLIT, dict(n=520, seqs=1, keys=1040)),
    (KSPLIT, dict(n=128, seqs=8, keys=144)),
    (NONE, dict(n=90, seqs=12, keys=144)),
    (KSPLIT, dict(n=90, seqs=12, keys=4112)),
    (NONE, dict(n=256, seqs=8, keys=272, D=64)),
    (NONE, dict(n=320, seqs=6, keys=336, D=64)),
    (KSPLIT, dict(n=321, seqs=5, keys=336, D=64)),
    (KSPLIT, dict(n=256, seqs=8, keys=4112, D=64)),
    (NONE, dict(n=119, seqs=5, keys=4112, total=357, D=64)),
    (KSPLIT, dict(n=119, seqs=5, keys=4112, D=64)),
    (NONE, dict(n=850, seqs=1, keys=1040, heads=24)),
    (KSPLIT, dict(n=850, seqs=1, keys=4112, heads=24)),
])
def test_pick_of_small_launches(want, kw):
    assert pick(**kw) == want
