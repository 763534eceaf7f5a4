"""Prompt attention with two items of a request to a workgroup and keys through LDS
(attention_block_kernel; grids of more workgroups than CUs): odd numbers of items, items of
one query, contexts at the edges of its 128-key stages, tree masks over two items, and
decode steps of more (request, head) pairs than CUs, against the oracle's rows and against
one workgroup per item."""
import ctypes

import numpy as np
import pytest

import flexflow_amd.ffmi as F
import test_gpu_kernels as K
from test_gpu_kernels import AttnCase, tree_masks

pytestmark = pytest.mark.gpu


def setup_module(module):
    K.setup_module(K)


def both(scenario, monkeypatch):
    blocks = scenario(True)
    monkeypatch.setenv("FFMI_ATTN_BLOCK", "0")
    single = scenario(False)
    for a, b in zip(blocks, single):
        a, b = a.astype(np.float32), b.astype(np.float32)
        # one rounding to fp16 of two fp32 sums of at most 1100 terms in other orders
        assert (np.abs(a - b) <= 2.0 ** -10 * np.abs(b) + 2e-6).all()
        assert (a == b).mean() > 0.97


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("steps", [[{0: 1, 1: 64, 2: 33, 3: 127, 4: 1, 5: 321}, {5: 95, 0: 250, 2: 7, 3: 2}],
                                   [{1: 600}, {1: 425, 0: 128}], [{2: 1023, 3: 1}, {3: 300, 2: 40, 1: 257}]])
@pytest.mark.parametrize("layout", [0, 1])
def test_prompt_blocks(d, steps, layout, monkeypatch):
    def scenario(oracle):
        rng = np.random.default_rng(d)
        c = AttnCase(F.ATTN_INC, heads=32, d=d, max_requests=6, max_seq=1100, max_tokens=1024,
                     out_layout=layout)
        done, res, got, want = {}, [], [], []
        for step in steps:
            infos = []
            for r, n in step.items():
                a = done.get(r, 0)
                infos += [(3, p, r, p, p + 1, 0, 0, 0) for p in range(a, a + n)]
                done[r] = a + n
            out, qs = c.run(infos, rng=rng)
            res.append(out[:len(infos)].copy())
            if oracle:
                for t in rng.choice(len(infos), size=12, replace=False):
                    got.append(out[t])
                    want.append(c.ref_row(qs[t], infos[t][2], range(infos[t][1] + 1)))
            else:
                rng.choice(len(infos), size=12, replace=False)
        if oracle:
            c.check(np.stack(got), np.stack(want))
        return res

    both(scenario, monkeypatch)


@pytest.mark.parametrize("d", [64, 128])
def test_tree_over_two_items(d, monkeypatch):
    def scenario(oracle):
        rng = np.random.default_rng(d + 1)
        R, n, depth0 = 9, 45, 100
        c = AttnCase(F.ATTN_TREE, heads=16, d=d, max_requests=R, max_seq=256, tree=64, max_tokens=1024)
        c.run([(3, p, r, p, p + 1, 0, 0, 0) for r in range(R) for p in range(depth0)], masks=[[0]] * R, rng=rng)
        parents = [-1] + [int(rng.integers(0, j)) for j in range(1, n)]
        m, depth = tree_masks(parents), [depth0]
        for j in range(1, n):
            depth.append(depth[parents[j]] + 1)
        infos = [(4, depth[j], r, depth0 + j, depth0, depth0, n, j) for r in range(R) for j in range(n)]
        out, qs = c.run(infos, masks=[m] * R, rng=rng)
        if oracle:
            rows = [5, 31, 32, n - 1, n + 33, 8 * n + 40]
            want = []
            for t in rows:
                anc, a = [], t % n
                while a >= 0:
                    anc.append(depth0 + a)
                    a = parents[a]
                want.append(c.ref_row(qs[t], t // n, list(range(depth0)) + sorted(anc)))
            c.check(out[rows], np.stack(want))
        return [out[:len(infos)].copy()]

    both(scenario, monkeypatch)


@pytest.mark.parametrize("d", [32, 64, 128])
def test_decode_of_many_pairs(d):
    rng = np.random.default_rng(d + 2)
    lens = [1, 31, 32, 33, 127, 128, 129, 160, 7]
    c = AttnCase(F.ATTN_INC, heads=32, d=d, max_requests=9, max_seq=256, max_tokens=1024)
    c.run([(3, p, r, p, p + 1, 0, 0, 0) for r, n in enumerate(lens) for p in range(n)], rng=rng)
    for step in range(2):
        infos = [(7, n + step, r, n + step, n + step + 1, 0, 0, 0) for r, n in enumerate(lens)]
        out, qs = c.run(infos, rng=rng)
        c.check(out[:9], np.stack([c.ref_row(qs[t], t, range(i[1] + 1)) for t, i in enumerate(infos)]))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("empty", [[], [(0, 288, 0, 0)], [(0, 288, 0, 288), (1, 288, 0, 0)], [(1, 288, 0, 40)]])
def test_items_without_queries(d, empty):
    """Items of no query behind the last row of a full batch, in a block of their own or as
    another's second: nothing of theirs is read or written."""
    T, L = 288, K.L
    c = AttnCase(F.ATTN_INC, heads=32, d=d, max_requests=2, max_seq=320, max_tokens=T)
    rng = np.random.default_rng(d)
    toks = (F.TokenInfo * T)(*[F.TokenInfo(3, p, 0, p, p + 1, 0, 0, 0, 0) for p in range(T)])
    qkv, got = K.Buf(K.f16(rng.standard_normal((T, 3 * c.Hl)))), []
    for extra in ([], empty):
        items = [(0, p, 32, p + 32) for p in range(0, T, 32)] + extra
        desc = F.BatchDesc(T, len(items), 0, 0, toks, (F.AttnWork * len(items))(*[F.AttnWork(*i) for i in items]),
                           (F.CommitInfo * 1)(), (ctypes.c_uint64 * 1)())
        F.check(L.ffmi_batch_upload(c.b, ctypes.byref(desc), None))
        out = K.Buf(np.full((T + 16, c.Hl), np.nan, np.float16))
        F.check(L.ffmi_attn_inc(c.h, c.b, qkv.ptr, out.ptr, None))
        got.append(out.get())
        assert np.isfinite(got[-1][:T]).all() and np.isnan(got[-1][T:]).all()
    assert np.array_equal(got[0].view(np.uint16), got[1].view(np.uint16))
