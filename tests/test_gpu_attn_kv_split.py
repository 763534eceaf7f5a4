"""Decode attention whose keys several workgroups share (attn_kv_split): at the edges of
its chunks (32 keys, 8 waves), with requests far shorter than the longest one (workgroups
without a key), in several steps on one handle (the counts return to zero), against one
workgroup per item and the oracle's rows."""
import ctypes

import numpy as np
import pytest

import flexflow_amd.ffmi as F
import test_gpu_kernels as K
from test_gpu_kernels import AttnCase, hip

pytestmark = pytest.mark.gpu


def setup_module(module):
    K.setup_module(K)


def caches(c):
    k, v, slots = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_int()
    F.check(K.L.ffmi_attn_kv_ptrs(c.h, ctypes.byref(k), ctypes.byref(v), ctypes.byref(slots)))
    out = np.empty((2, 4 * c.heads * slots.value * c.d), np.uint16)
    for row, p in zip(out, (k, v)):
        hip().hipMemcpy(row.ctypes.data, p, row.nbytes, 2)
    return out


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("lens", [[255], [256], [511, 3, 300], [513, 512, 40, 257], [1793, 1], [2080],
                                  [1279, 1, 1280]])
@pytest.mark.parametrize("layout", [0, 1])
def test_split_keys(d, lens, layout, monkeypatch):
    def scenario(oracle):
        rng = np.random.default_rng(d + len(lens))
        c = AttnCase(F.ATTN_INC, d=d, max_seq=2176, max_tokens=1024, out_layout=layout)
        for r, n in enumerate(lens):
            for a in range(0, n, 1024):
                c.run([(3, p, r, p, p + 1, 0, 0, 0) for p in range(a, min(n, a + 1024))], rng=rng)
        got, want = [], []
        for step in range(3):
            infos = [(7, n + step, r, n + step, n + step + 1, 0, 0, 0) for r, n in enumerate(lens)]
            out, qs = c.run(infos, rng=rng)
            got.append(out[:len(lens)])
            if oracle:
                want.append(np.stack([c.ref_row(qs[t], t, range(i[1] + 1)) for t, i in enumerate(infos)]))
        if oracle:
            c.check(np.concatenate(got), np.concatenate(want))
        return np.concatenate(got).astype(np.float32), caches(c)

    split, kv = scenario(True)
    monkeypatch.setenv("FFMI_ATTN_KVSPLIT", "0")
    whole, kv1 = scenario(False)
    assert np.array_equal(kv, kv1)
    # one rounding to fp16 of two fp32 sums of at most 2083 terms in other orders
    assert (np.abs(split - whole) <= 2.0 ** -10 * np.abs(whole) + 2e-6).all()
    assert (split == whole).mean() > 0.97


def step_on(c, batch, stream, infos, qkv, out):
    """One decode step of c's handle on a stream, from a batch of its own."""
    toks = (F.TokenInfo * len(infos))(*[F.TokenInfo(*i, 0) for i in infos])
    work = (F.AttnWork * len(infos))(*[F.AttnWork(i[2], t, 1, i[4]) for t, i in enumerate(infos)])
    desc = F.BatchDesc(len(infos), len(infos), 0, 0, toks, work, (F.CommitInfo * 1)(), (ctypes.c_uint64 * 1)())
    F.check(K.L.ffmi_batch_upload(batch, ctypes.byref(desc), stream))
    F.check(K.L.ffmi_attn_inc(c.h, batch, qkv.ptr, out.ptr, stream))


@pytest.mark.parametrize("heads,lens", [(2, [2080, 700, 1300, 400]), (16, [1025, 513, 2000, 300])])
def test_two_streams_on_one_handle(heads, lens):
    """Steps of different requests side by side: splits of different widths (the first
    request alone, the other three together) count for themselves."""
    d, H = 128, hip()
    c = AttnCase(F.ATTN_INC, heads=heads, d=d, max_seq=2176, max_tokens=1024)
    rng = np.random.default_rng(heads)
    for r, n in enumerate(lens):
        for a in range(0, n, 1024):
            c.run([(3, p, r, p, p + 1, 0, 0, 0) for p in range(a, min(n, a + 1024))], rng=rng)
    groups, sides = [[0], [1, 2, 3]], []
    for g in groups:
        b, s = ctypes.c_void_p(), ctypes.c_void_p()
        F.check(K.L.ffmi_batch_create(64, 4, ctypes.byref(b)))
        assert H.hipStreamCreate(ctypes.byref(s)) == 0
        infos = [(7, lens[r], r, lens[r], lens[r] + 1, 0, 0, 0) for r in g]
        qkv = K.Buf(K.f16(rng.standard_normal((len(g), 3 * c.Hl))))
        sides.append((b, s, infos, qkv, [K.Buf.empty((16, c.Hl), np.float16) for _ in range(41)]))
    for b, s, infos, qkv, outs in sides:  # one after the other
        step_on(c, b, s, infos, qkv, outs[0])
        assert H.hipStreamSynchronize(s) == 0
    for i in range(1, 41):  # side by side, the same step again and again
        for b, s, infos, qkv, outs in sides:
            step_on(c, b, s, infos, qkv, outs[i])
    for _, s, _, _, _ in sides:
        assert H.hipStreamSynchronize(s) == 0
    for g, (b, s, infos, qkv, outs) in zip(groups, sides):
        want = outs[0].get()[:len(g)].view(np.uint16)
        assert want.any()
        for o in outs[1:]:
            assert np.array_equal(o.get()[:len(g)].view(np.uint16), want)


def test_one_request_in_two_items():
    """A request's keys are split where one item has them: with the request in two items
    (apart, over keys of earlier steps) each has a workgroup of its own."""
    d, n, L = 128, 900, K.L
    c = AttnCase(F.ATTN_INC, heads=2, d=d, max_seq=1024, max_tokens=1024)
    rng = np.random.default_rng(5)
    for r in (0, 1):
        c.run([(3, p, r, p, p + 1, 0, 0, 0) for p in range(n)], rng=rng)
    qkv, outs = K.Buf(K.f16(rng.standard_normal((3, 3 * c.Hl)))), []
    for reqs in ((0, 1, 0), (0, 1)):
        infos = [(7, n - 1, r, -1, n, 0, 0, 0) for r in reqs]  # (nothing is stored)
        out = K.Buf(np.full((16, c.Hl), np.nan, np.float16))
        step_on(c, c.b, None, infos, qkv, out)
        outs.append(out.get()[:len(reqs)].astype(np.float32))
        assert np.isfinite(outs[-1]).all()
    # shared and unshared keys: the other order of sums, one rounding to fp16
    assert (np.abs(outs[0][:2] - outs[1]) <= 2.0 ** -10 * np.abs(outs[1]) + 2e-6).all()
    # the third row is another query of the first request
    assert not np.array_equal(outs[0][0], outs[0][2])
