"""Decode steps whose products norm their own operands (up to 16 tokens, 2048 to 4096 channels; the
residual in packed tiles, the norm weight in LDS) against steps with norm launches."""
import numpy as np
import pytest

import flexflow_amd as fa
from flexflow_amd import ffmi as F
from hip_util import Buf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,heads", [(2048, 16), (2112, 33), (4096, 32), (4160, 65)])
def test_steps(monkeypatch, hidden, heads):
    """Where the sum of squares is taken in another order, a row's rms may round the other way, and so may
    its products; products of 2048 columns are split over K beside norm launches alone."""
    cfg = dict(num_layers=2, vocab_size=500, num_heads=heads, num_kv_heads=heads, hidden=hidden, intermediate=288,
               rms_eps=1e-6, rope_theta=10000.0)
    seq = np.random.default_rng(3).integers(0, 500, 120).tolist()
    out = []
    for mode in ("1", "0"):
        monkeypatch.setenv("FFMI_FUSE_NORM", mode)
        m = fa.Model(cfg, "inc", max_requests=2, max_tokens=64, max_seq_len=128, weight_seed=7)
        rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_sequence_length=128)
        parts, at = [], 0
        for k in (3, 1, 2, 8, 15, 16, 17, 32, 7):
            parts.append(rm.replay_step(m, [(1, seq[at:at + k], range(k))]))
            at += k
        out.append(np.concatenate(parts))
    # a rounding of a product's operands (2^-11 each, of either sign) moves a row by 2^-11 of its 2-norm:
    # four norms in two layers; an element by four times its row's root mean square of that
    d, rms = np.abs(out[0] - out[1]), np.sqrt((out[1] ** 2).mean(1, keepdims=True))
    assert (np.sqrt((d * d).mean(1, keepdims=True)) <= 4 * 2.0 ** -11 * rms).all()
    assert (d <= 16 * 2.0 ** -11 * rms).all()


def half(rng, *shape, scale=1.0):
    return (rng.standard_normal(shape) * scale).astype(np.float16)


def pack(L, w):
    src, dst = Buf(w), Buf.empty((L.ffmi_linear_packed_bytes(*w.shape) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_weight(src.ptr, *w.shape, dst.ptr, None))
    return dst


def pack_rows(L, x):
    src, dst = Buf(x), Buf.empty((L.ffmi_packed_activation_bytes(*x.shape) // 2,), np.uint16)
    F.check(L.ffmi_pack_activations(src.ptr, *x.shape, dst.ptr, None))
    return dst


@pytest.mark.parametrize("stream", [0, F.W_STREAM])
@pytest.mark.parametrize("H,K,N,gated", [(4096, 4096, 12288, False), (4096, 320, 11008, True), (2048, 5632, 6144, False),
                                         (64, 64, 256, False), (96, 64, 256, True), (2080, 96, 256, False)])
def test_packed_and_in_rows_the_same_bits(H, K, N, gated, stream):
    """The pair as models run it, operands and residual in packed tiles, against rows; waves with no
    k-step of their own (64 and 96 channels) and with a batch and a rest (2080)."""
    L, rng = F.lib(), np.random.default_rng(H + N)
    wo, wn = pack(L, half(rng, H, K, scale=0.02)), Buf(1 + half(rng, H, scale=0.1))
    if gated:
        parts = [Buf(half(rng, N, H, scale=0.02)) for _ in range(2)]
        w = Buf.empty((L.ffmi_linear_packed_bytes(N, H),), np.uint16)
        F.check(L.ffmi_linear_pack_gate_up(parts[0].ptr, parts[1].ptr, N, H, w.ptr, None))
    else:
        w = pack(L, half(rng, N, H, scale=0.02))
    epi = (F.EPI_SILU_MUL if gated else F.EPI_NONE) | stream
    for T in (1, 5, 8, 15, 16):
        x, r = half(rng, T, K), half(rng, T, H)
        xb, xp, res, ss, y = Buf(x), pack_rows(L, x), Buf(r), Buf.empty((T, H // 16), np.float32), \
            Buf.empty((T, N), np.float16)
        packed = Buf.empty((L.ffmi_packed_activation_bytes(T, H) // 2,), np.uint16)
        F.check(L.ffmi_debug_fused_residual_linear_packed(xb.ptr, wo.ptr, res.ptr, packed.ptr, ss.ptr, T, H, K,
                                                          stream, None))
        F.check(L.ffmi_debug_fused_norm_linear(res.ptr, ss.ptr, wn.ptr, 1e-6, w.ptr, y.ptr, T, N, H, epi, None))
        want = res.get(), ss.get(), y.get()
        res, ss, y = Buf(r), Buf.empty((T, H // 16), np.float32), Buf.empty((T, N), np.float16)
        F.check(L.ffmi_debug_fused_residual_linear_packed(xp.ptr, wo.ptr, res.ptr, packed.ptr, ss.ptr, T, H, K,
                                                          F.X_PACKED | stream, None))
        F.check(L.ffmi_debug_fused_norm_linear(packed.ptr, ss.ptr, wn.ptr, 1e-6, w.ptr, y.ptr, T, N, H,
                                               F.X_PACKED | epi, None))
        for got, ref in zip((res.get(), ss.get(), y.get()), want):
            assert np.isfinite(ref.astype(np.float32)).all() and np.array_equal(got, ref), T
        if not stream:  # and the rows of the form without packed tiles
            res, ss = Buf(r), Buf.empty((T, H // 16), np.float32)
            F.check(L.ffmi_debug_fused_residual_linear(xb.ptr, wo.ptr, res.ptr, ss.ptr, T, H, K, None))
            assert np.array_equal(res.get(), want[0]) and np.array_equal(ss.get(), want[1]), T
