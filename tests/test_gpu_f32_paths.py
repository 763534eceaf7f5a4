"""Full-precision kernels at the edges of their forms: the linear layer's tile forms against
the path for unaligned rows (the same order of sums, so bit for bit) and an fp64 product; the
norm's widths and its path for rows that are not of 16-byte pieces; the attention around its
passes of 32 and 128 keys."""
import ctypes

import numpy as np
import pytest

import flexflow_amd as fa
import flexflow_amd.ffmi as F
import oracle_lib as O
import test_gpu_kernels as K
from hip_util import Buf
from test_gpu_kernels import AttnCase

pytestmark = pytest.mark.gpu


def setup_module(module):
    K.setup_module(K)


class Array:
    """fp32 values on the device, `skip` elements into a buffer with one more behind."""

    def __init__(self, x, skip=0):
        x = np.asarray(x, np.float32)
        self.buf, self.skip, self.shape = Buf(np.concatenate([np.full(skip, 7), x.ravel(), [7]]).astype(np.float32)), \
            skip, x.shape
        self.ptr = ctypes.c_void_p(self.buf.ptr.value + 4 * skip)

    def get(self):
        x = self.buf.get()
        assert (x[:self.skip] == 7).all() and x[-1] == 7  # nothing written outside
        return x[self.skip:-1].reshape(self.shape)


@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 48, 64, 65, 96, 97, 129, 201, 300])
@pytest.mark.parametrize("N,k", [(16, 32), (100, 96), (2050, 160), (9000, 64), (768, 1056)])
def test_linear_forms(T, N, k):
    rng = np.random.default_rng(T)
    x, w = rng.standard_normal((T, k)).astype(np.float32), rng.standard_normal((N, k)).astype(np.float32)
    got = []
    for skip in (0, 1):
        xd, wd, y = Array(x, skip), Array(w, skip), Array(np.zeros((T, N)), skip)
        F.check(K.L.ffmi_linear_f32(xd.ptr, wd.ptr, y.ptr, T, N, k, None))
        got.append(y.get())
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    ref, mag = x.astype(np.float64) @ w.astype(np.float64).T, np.abs(x) @ np.abs(w).T
    assert (np.abs(got[0] - ref) <= 2e-6 * mag + 1e-30).all()


# both sides of the lines between registers and rings of two and of four k-blocks
@pytest.mark.parametrize("T,N,k", [(4, 100, 256), (5, 100, 256), (4, 100, 288), (16, 2050, 512), (16, 2050, 544),
                                   (3, 4096, 1024), (3, 4095, 1024), (16, 4100, 1056)])
def test_linear_of_few_rows(T, N, k):
    test_linear_forms(T, N, k)


@pytest.mark.parametrize("H", [4, 102, 1020, 1024, 1028, 2048, 4096, 8192, 8196])
@pytest.mark.parametrize("form", ["plain", "residual", "alias", "unaligned"])
def test_norm_widths(H, form):
    rng = np.random.default_rng(H)
    T, eps, skip = 3, 1e-6, int(form == "unaligned")
    x1, x2, w = (rng.standard_normal(n).astype(np.float32) for n in ((T, H), (T, H), (H,)))
    r = x1 if form == "plain" else x1 + x2
    a, b, wd, out = Array(x1, skip), Array(x2, skip), Array(w, skip), Array(np.zeros((T, H)), skip)
    if form == "plain":
        F.check(K.L.ffmi_rmsnorm_f32(a.ptr, wd.ptr, out.ptr, T, H, eps, None))
    else:
        res = a if form == "alias" else Array(np.zeros((T, H)), skip)
        F.check(K.L.ffmi_residual_rmsnorm_f32(a.ptr, b.ptr, wd.ptr, res.ptr, out.ptr, T, H, eps, None))
        assert np.array_equal(res.get(), r)
    r = r.astype(np.float64)
    ref = r / np.sqrt((r * r).mean(1, keepdims=True) + np.float32(eps)) * w.astype(np.float64)
    # sum / H, + eps, sqrt, 1 / and two products: at most half an ulp each
    assert (np.abs(out.get() - ref) <= 6 * 2.0 ** -24 * np.abs(ref)).all()


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("lens", [{0: 1, 1: 31}, {0: 32, 1: 33, 2: 127}, {0: 128, 1: 129, 3: 160}])
def test_attention_passes(d, lens):
    rng = np.random.default_rng(d + sum(lens.values()))
    c = AttnCase(F.ATTN_INC, d=d, max_seq=256, max_tokens=512, fp32=True)
    c.run([(3, p, r, p, p + 1, 0, 0, 0) for r, n in lens.items() for p in range(n)], rng=rng)
    infos = [(7, n, r, n, n + 1, 0, 0, 0) for r, n in lens.items()]
    out, qs = c.run(infos, rng=rng)
    c.check(out[:len(infos)], np.stack([c.ref_row(qs[t], i[2], range(i[1] + 1)) for t, i in enumerate(infos)]))


# outputs in the queries' own buffer, from its start or overlapping its end: as in a buffer of their own
@pytest.mark.parametrize("at", [0, 1, 2])
def test_attention_output_in_its_input(at):
    T, c = 4, AttnCase(F.ATTN_INC, heads=8, d=128, max_seq=256, max_tokens=512, fp32=True)
    c.run([(3, p, r, p, p + 1, 0, 0, 0) for r in range(T) for p in range(40 + r)], rng=np.random.default_rng(1))
    want, _ = c.run([(7, 40 + r, r, 40 + r, 41 + r, 0, 0, 0) for r in range(T)], rng=np.random.default_rng(2))
    qkv = np.random.default_rng(2).standard_normal((T, 3 * c.Hl)).astype(np.float32)
    off = (0, 5, 3 * T - 1)[at] * c.Hl
    buf = Buf(np.concatenate([qkv.ravel(), np.zeros(T * c.Hl, np.float32)]))
    F.check(K.L.ffmi_attn_inc(c.h, c.b, buf.ptr, ctypes.c_void_p(buf.ptr.value + 4 * off), None))
    got = buf.get()[off:off + T * c.Hl].reshape(T, c.Hl)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("heads", [128, 129])
def test_first_norm_of_wide_rows(heads):
    """A step's first norm gathers the tokens' rows and brings the step's blob to the device; rows of
    more than 8192 columns take a copy and the scalar kernel.  Steps of several requests, whose
    tokens lie elsewhere in the blob; 2-norm within 8192 terms' roundings of 2^-24."""
    cfg = dict(num_layers=1, vocab_size=64, num_heads=heads, num_kv_heads=heads, hidden=64 * heads, intermediate=32,
               rms_eps=1e-6, rope_theta=10000.0)
    m = fa.Model(cfg, "inc", max_requests=3, max_tokens=64, max_seq_len=64, weight_seed=11, full_precision=True)
    rm = fa.RequestManager(max_requests_per_batch=3, max_tokens_per_batch=64, max_spec_tree_token_num=0,
                           max_sequence_length=64)
    ref = O.Model(cfg, 11, fp16=0, max_requests=3, max_seq=64)
    rng = np.random.default_rng(heads)
    toks, at, got = rng.integers(0, 64, (3, 40)), [0, 0, 0], [[], [], []]
    for step in ((5, 0, 0), (1, 7, 0), (1, 1, 20), (1, 1, 1), (17, 1, 1)):
        part = [(r + 1, toks[r][at[r]:at[r] + n], range(n)) for r, n in enumerate(step) if n]
        rows = np.split(rm.replay_step(m, part), np.cumsum([n for n in step if n])[:-1])
        for r in (r for r in range(3) if step[r]):
            got[r].append(rows.pop(0))
            at[r] += step[r]
    for r in range(3):
        want = ref.forward(r, toks[r][:at[r]].astype(np.int32), 0)
        d = np.linalg.norm(np.concatenate(got[r]) - want, axis=1) / np.linalg.norm(want, axis=1)
        assert (d <= 8192 ** 0.5 * 2.0 ** -24 * 4).all(), d.max()
