"""Dense layers on row-major activations that the library packs first (api.cpp pack_first):
the same bits as activations packed by the caller, with a workspace that has no room for
them, and in a captured graph."""
import ctypes

import numpy as np
import pytest

import flexflow_amd.ffmi as F
import test_gpu_kernels as K
from hip_util import Buf, f16, hip, sync

pytestmark = pytest.mark.gpu


def setup_module(module):
    K.setup_module(K)


@pytest.mark.parametrize("T,N,k,epi", [(129, 9700, 2080, 0), (168, 4096, 4096, 0), (200, 2912, 2208, 1),
                                       (193, 15000, 992, 0), (128, 9700, 2080, 0), (300, 1000, 4128, 1)])
def test_row_major(T, N, k, epi):
    L, H = K.L, hip()
    rng = np.random.default_rng(T)
    X, W = f16(rng.standard_normal((T, k))), [Buf(f16(rng.uniform(-0.05, 0.05, (N, k)))) for _ in range(1 + epi)]
    Wp = Buf.empty(((1 + epi) * L.ffmi_linear_packed_bytes(N, k) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_gate_up(W[0].ptr, W[1].ptr, N, k, Wp.ptr, None) if epi else
            L.ffmi_linear_pack_weight(W[0].ptr, N, k, Wp.ptr, None))
    Xb, Xp = Buf(X), Buf.empty((L.ffmi_packed_activation_bytes(T, k) // 2,), np.uint16)
    F.check(L.ffmi_pack_activations(Xb.ptr, T, k, Xp.ptr, None))
    want = Buf.empty((T, N), np.float16)
    F.check(L.ffmi_linear(Xp.ptr, Wp.ptr, want.ptr, T, N, k, epi | F.X_PACKED, None))
    want = want.get().view(np.uint16)

    def fresh():
        return Buf(np.full((T, N), np.nan, np.float16))
    y = fresh()
    F.check(L.ffmi_linear(Xb.ptr, Wp.ptr, y.ptr, T, N, k, epi, None))
    assert np.array_equal(y.get().view(np.uint16), want)
    # the caller's workspace: all of it, and the slabs alone
    for flags in (epi, epi | F.X_PACKED):
        n = L.ffmi_linear_workspace_bytes(T, N, k, flags)
        ws, y = Buf.empty((max(n, 16),), np.uint8), fresh()
        F.check(L.ffmi_linear_ws(Xb.ptr, Wp.ptr, y.ptr, T, N, k, epi, ws.ptr, n, None))
        assert np.array_equal(y.get().view(np.uint16), want)
    # captured, and replayed after the library's workspace was used by others
    s, g, ex, y = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p(), fresh()
    assert H.hipStreamCreate(ctypes.byref(s)) == 0
    sync()
    assert H.hipStreamBeginCapture(s, 2) == 0
    F.check(L.ffmi_linear(Xb.ptr, Wp.ptr, y.ptr, T, N, k, epi, s))
    assert H.hipStreamEndCapture(s, ctypes.byref(g)) == 0
    assert H.hipGraphInstantiate(ctypes.byref(ex), g, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        F.check(L.ffmi_linear(Xb.ptr, Wp.ptr, fresh().ptr, T, N, k, epi, None))
        sync()
        assert H.hipGraphLaunch(ex, s) == 0
        assert H.hipStreamSynchronize(s) == 0
        assert np.array_equal(y.get().view(np.uint16), want)
    H.hipGraphExecDestroy(ex), H.hipGraphDestroy(g)


# products that the tile kernel takes row-major and the M-split kernel packed (short
# slices), and shorter ones that are packed first
@pytest.mark.parametrize("T,N,k,epi", [(300, 2304, 768, 0), (257, 512, 4096, 0), (384, 2816, 1024, 1), (300, 1000, 256, 0),
                                       (350, 72, 4096, 0), (257, 2040, 2080, 0), (270, 1000, 1024, 0), (193, 768, 768, 0)])
def test_row_major_of_few_steps(T, N, k, epi):
    test_row_major(T, N, k, epi)


@pytest.mark.parametrize("T", [1, 3, 8, 9, 15, 16, 17, 24, 33, 64])
@pytest.mark.parametrize("epi", [0, 1])
def test_packed_rows_past_the_last(T, epi):
    """Packed activations of few rows: what lies in the last tile's other rows is not
    computed with (the row-major layout has none, and gives the same bits)."""
    L, N, k = K.L, 1000, 1088
    rng = np.random.default_rng(T)
    X, W = f16(rng.standard_normal((T, k))), [Buf(f16(rng.uniform(-0.05, 0.05, (N, k)))) for _ in range(2)]
    Wp = Buf.empty(((1 + epi) * L.ffmi_linear_packed_bytes(N, k) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_gate_up(W[0].ptr, W[1].ptr, N, k, Wp.ptr, None) if epi else
            L.ffmi_linear_pack_weight(W[0].ptr, N, k, Wp.ptr, None))
    pad = f16(np.concatenate([X.astype(np.float32), np.full((-T % 16, k), np.nan, np.float32)]))
    got = []
    for x, flags in ((Buf(X), 0), (Buf(K.pack_act_np(pad)), F.X_PACKED)):
        y = Buf(np.full((T, N), np.nan, np.float16))
        F.check(L.ffmi_linear(x.ptr, Wp.ptr, y.ptr, T, N, k, epi | flags, None))
        got.append(y.get().view(np.uint16))
    assert np.array_equal(*got)


@pytest.mark.parametrize("T,N,k", [(200, 704, 1024), (300, 2050, 256), (200, 4100, 4096), (40, 704, 1024)])
def test_buffers_off_16_bytes(T, N, k):
    """Activations and a workspace that are both 4 bytes off a 16-byte boundary: the forms
    that load them as they are."""
    L = K.L
    rng = np.random.default_rng(T)
    X, W = f16(rng.standard_normal((T, k))), Buf(f16(rng.uniform(-0.05, 0.05, (N, k))))
    Wp = Buf.empty((L.ffmi_linear_packed_bytes(N, k) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_weight(W.ptr, N, k, Wp.ptr, None))
    n, got = L.ffmi_linear_workspace_bytes(T, N, k, 0), []
    for off in (0, 4):
        x = Buf(np.concatenate([np.zeros(off // 2, np.float16), X.ravel().view(np.float16), np.zeros(8, np.float16)]))
        y, ws = Buf(np.full((T, N), np.nan, np.float16)), Buf.empty((n + 64,), np.uint8)
        F.check(L.ffmi_linear_ws(ctypes.c_void_p(x.ptr.value + off), Wp.ptr, y.ptr, T, N, k, 0,
                                 ctypes.c_void_p(ws.ptr.value + off), n, None))
        got.append(y.get())
    K.close16(got[1], got[0].astype(np.float32))


@pytest.mark.parametrize("off_x,off_ws", [(4, 0), (2, 0), (0, 4), (4, 4)])
@pytest.mark.parametrize("T,N,k", [(200, 4100, 4096), (300, 3000, 288)])
def test_one_buffer_off_16_bytes(T, N, k, off_x, off_ws):
    """Each by itself: activations off a 16-byte boundary are packed as others are (the pass
    loads them as they lie) where the workspace is on one, and a workspace that is off one
    holds slabs alone."""
    L = K.L
    rng = np.random.default_rng(T + off_x)
    X, W = f16(rng.standard_normal((T, k))), Buf(f16(rng.uniform(-0.05, 0.05, (N, k))))
    Wp = Buf.empty((L.ffmi_linear_packed_bytes(N, k) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_weight(W.ptr, N, k, Wp.ptr, None))
    n, got = L.ffmi_linear_workspace_bytes(T, N, k, 0), []
    for ox, ow in ((0, 0), (off_x, off_ws)):
        x = Buf(np.concatenate([np.zeros(ox // 2, np.float16), X.ravel().view(np.float16), np.zeros(8, np.float16)]))
        y, ws = Buf(np.full((T, N), np.nan, np.float16)), Buf.empty((n + 64,), np.uint8)
        F.check(L.ffmi_linear_ws(ctypes.c_void_p(x.ptr.value + ox), Wp.ptr, y.ptr, T, N, k, 0,
                                 ctypes.c_void_p(ws.ptr.value + ow), n, None))
        got.append(y.get())
    K.close16(got[1], got[0].astype(np.float32))
    if k == 4096 and not off_ws:  # packed both times
        assert np.array_equal(got[1].view(np.uint16), got[0].view(np.uint16))


@pytest.mark.parametrize("T,later", [(168, (168,)), (256, (257, 384))])
def test_graph_before_eager_growth(T, later):
    """A graph's slabs stay valid when eager calls after the capture ask the library's
    workspace for more: the same call (its packed activations), and longer ones."""
    L, H, N, k = K.L, hip(), 4096, 11008
    rng = np.random.default_rng(T)
    X, W = f16(rng.standard_normal((max(later), k))), Buf(f16(rng.uniform(-0.05, 0.05, (N, k))))
    Wp = Buf.empty((L.ffmi_linear_packed_bytes(N, k) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_weight(W.ptr, N, k, Wp.ptr, None))
    x, y = Buf(X), Buf(np.full((T, N), np.nan, np.float16))
    s, g, ex = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert H.hipStreamCreate(ctypes.byref(s)) == 0
    sync()
    assert H.hipStreamBeginCapture(s, 2) == 0
    F.check(L.ffmi_linear(x.ptr, Wp.ptr, y.ptr, T, N, k, 0, s))
    assert H.hipStreamEndCapture(s, ctypes.byref(g)) == 0
    assert H.hipGraphInstantiate(ctypes.byref(ex), g, None, None, ctypes.c_size_t(0)) == 0
    z = Buf(np.full((max(later), N), np.nan, np.float16))
    for t in (*later, T):
        F.check(L.ffmi_linear(x.ptr, Wp.ptr, z.ptr, t, N, k, 0, None))
        sync()
        # whoever is given memory now keeps what is written there
        others = [Buf(np.full((n << 20,), 7, np.uint8)) for n in (8, 22, 26, 34)]
        assert H.hipGraphLaunch(ex, s) == 0
        assert H.hipStreamSynchronize(s) == 0
        assert all((b.get() == 7).all() for b in others)
    assert np.array_equal(y.get().view(np.uint16), z.get()[:T].view(np.uint16))
    H.hipGraphExecDestroy(ex), H.hipGraphDestroy(g)
