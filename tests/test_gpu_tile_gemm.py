"""The tile form of the dense layers (gemm_tile_kernel, T > 64) where it can go
wrong: rows and columns past a tile's edge, fewer k-steps than ring stages, every
tile size by itself and in K slices summed by the reduce pass, row-major and packed
activations, both epilogues.
Tolerance as test_gpu_kernels.close16."""
import ctypes
import zlib

import numpy as np
import pytest

import flexflow_amd.ffmi as F
import oracle_lib as O
from hip_util import Buf, f16
from test_gpu_kernels import close16, pack_act_np, unpack_act_np

pytestmark = pytest.mark.gpu

# (T, N, K): small ones with one to a few k-steps, then what the plan gives most tile
# sizes (FORMS has the others)
CASES = [(65, 8, 32), (129, 40, 64), (193, 136, 96), (257, 72, 160), (513, 264, 288),
         (170, 2040, 2048), (161, 4104, 4096), (1009, 4104, 1024), (1009, 6152, 1024), (377, 5624, 1024),
         (529, 12296, 1024), (241, 20008, 1024), (1009, 12296, 1024), (313, 20008, 1024), (849, 20008, 1024)]


@pytest.mark.parametrize("epi", [0, 1])
@pytest.mark.parametrize("T,N,K", CASES)
def test_tile_edges(T, N, K, epi, monkeypatch):
    if epi and N > 8000:
        N //= 2
    N += -N % 32 if epi else 0  # (packed outputs are whole k-steps wide)
    monkeypatch.setenv("FFMI_TILE_GEMM", "2")
    L = F.lib()
    rng = np.random.default_rng(zlib.crc32(f"{T}:{N}:{K}:{epi}".encode()))
    X = f16(rng.standard_normal((T, K)))
    W = f16(rng.uniform(-0.05, 0.05, ((2 if epi else 1) * N, K)))
    Wp = Buf.empty(((2 if epi else 1) * L.ffmi_linear_packed_bytes(N, K) // 2,), np.uint16)
    if epi:
        gb, ub = Buf(np.ascontiguousarray(W[:N])), Buf(np.ascontiguousarray(W[N:]))
        F.check(L.ffmi_linear_pack_gate_up(gb.ptr, ub.ptr, N, K, Wp.ptr, None))
    else:
        src = Buf(W)
        F.check(L.ffmi_linear_pack_weight(src.ptr, N, K, Wp.ptr, None))
    Xr, Xp = Buf(X), Buf(pack_act_np(X))
    Y = Buf.empty((T + 1, N), np.float16)  # (a row more: nothing may land there)
    F.check(L.ffmi_linear(Xr.ptr, Wp.ptr, Y.ptr, T, N, K, epi, None))
    y = Y.get()
    assert not y[T].any()
    Z = Buf.empty((T + 1, N), np.float16)
    F.check(L.ffmi_linear(Xp.ptr, Wp.ptr, Z.ptr, T, N, K, epi | F.X_PACKED, None))
    assert np.array_equal(Z.get().view(np.uint16), y.view(np.uint16))
    if epi:
        P = Buf.empty(((T + 15) // 16 * 16, N), np.float16)
        F.check(L.ffmi_linear(Xp.ptr, Wp.ptr, P.ptr, T, N, K, epi | F.X_PACKED | F.Y_PACKED, None))
        assert np.array_equal(unpack_act_np(P.get(), T, N).view(np.uint16), y[:T].view(np.uint16))
        # sums of another order may round g or u to the next fp16: the unit's slope is below
        # 1.1, so an output moves by at most 1.1 ulps of each factor's product
        g, u = (O.linear(X.astype(np.float32), w.astype(np.float32), fp16=1).astype(np.float64)
                for w in (W[:N], W[N:]))
        ref = g / (1.0 + np.exp(-g)) * u
        tol = 2.0 ** -9 * (np.abs(g) + 2.0 ** -4) * (np.abs(u) + 2.0 ** -4) + 1e-4 * np.abs(ref).max()
        assert (np.abs(y[:T] - ref) <= tol).all(), np.abs(y[:T] - ref).max()
    else:
        close16(y[:T], O.linear(X.astype(np.float32), W.astype(np.float32), fp16=1))


# (T, N, K, epilogue, form, in K slices): with CASES, every form in and out of slices, for
# both epilogues (test_linear_plans.py checks that), at remainders of rows and columns
FORMS = [(849, 10008, 512, 0, 7, False), (513, 20008, 288, 0, 8, False), (289, 8224, 2048, 1, 5, False),
         (193, 12320, 288, 1, 6, False), (513, 10016, 288, 1, 8, False),
         (193, 3000, 4096, 0, 2, True), (193, 5624, 5632, 0, 3, True), (129, 5624, 5632, 0, 4, True),
         (289, 4104, 8192, 0, 5, True), (193, 4104, 11008, 0, 6, True), (193, 8200, 11008, 0, 7, True),
         (129, 8200, 11008, 0, 8, True), (193, 12296, 8192, 0, 9, True),
         (65, 64, 1024, 1, 0, True), (65, 3008, 2048, 1, 1, True), (193, 1024, 11008, 1, 2, True),
         (193, 3008, 5632, 1, 3, True), (129, 3008, 8192, 1, 4, True), (289, 3008, 8192, 1, 5, True),
         (193, 4128, 5632, 1, 6, True), (193, 4128, 11008, 1, 7, True), (129, 8224, 4096, 1, 8, True),
         (193, 6176, 8192, 1, 9, True)]


@pytest.mark.parametrize("T,N,K,epi,form,sliced", FORMS)
def test_forms(T, N, K, epi, form, sliced, monkeypatch):
    monkeypatch.setenv("FFMI_TILE_GEMM", "2")
    slices = ctypes.c_int()
    assert F.lib().ffmi_debug_linear_tiles(T, N, K, epi, ctypes.byref(slices)) == form
    assert (slices.value > 1) == sliced
    test_tile_edges(T, N * 2 if epi and N > 8000 else N, K, epi, monkeypatch)  # (which halves such N)


# the sizes of one row block, in and out of K slices: the hint of a weight stream changes
# where the weights are kept, not what is computed
@pytest.mark.parametrize("T,N,K,epi,form", [(193, 4104, 11008, 0, 6), (200, 20008, 512, 0, 6), (193, 8200, 11008, 0, 7),
                                            (193, 12296, 8192, 0, 9), (200, 12320, 288, 1, 6), (193, 20032, 512, 1, 7),
                                            (193, 6176, 8192, 1, 9)])
def test_weight_stream(T, N, K, epi, form):
    L = F.lib()
    assert L.ffmi_debug_linear_tiles(T, N, K, epi, None) == form
    rng = np.random.default_rng(T)
    X = Buf(pack_act_np(f16(rng.standard_normal((T, K)))))
    W = [Buf(f16(rng.uniform(-0.05, 0.05, (N, K)))) for _ in range(1 + epi)]
    Wp = Buf.empty(((1 + epi) * L.ffmi_linear_packed_bytes(N, K) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_gate_up(W[0].ptr, W[1].ptr, N, K, Wp.ptr, None) if epi else
            L.ffmi_linear_pack_weight(W[0].ptr, N, K, Wp.ptr, None))
    got = []
    for hint in (0, F.W_STREAM):
        y = Buf(np.full((T + 1, N), np.nan, np.float16))
        F.check(L.ffmi_linear(X.ptr, Wp.ptr, y.ptr, T, N, K, epi | F.X_PACKED | hint, None))
        got.append(y.get())
        assert np.isfinite(got[-1][:T]).all() and np.isnan(got[-1][T]).all()
    assert np.array_equal(*(g[:T].view(np.uint16) for g in got))


# 65 .. 192 rows, 96 columns a workgroup: edges of the row tiles and of the two row counts,
# columns past the last whole tile of 96, one k-step to more than the ring's stages (and
# slices of K, another kernel's).  Row-major activations of these sizes take the M-split kernel, whose
# order of sums is the same.
TWELVE_ROWS = [65, 81, 128, 129, 176, 192]
TWELVE = [(16392, 32, 0), (20008, 96, 0), (16392, 160, 0), (16400, 512, 0), (8224, 32, 1), (11040, 288, 1),
          (4120, 2560, 0)]


@pytest.mark.parametrize("stream", [0, F.W_STREAM])
@pytest.mark.parametrize("T", TWELVE_ROWS)
@pytest.mark.parametrize("N,K,epi", TWELVE)
def test_twelve_waves(T, N, K, epi, stream):
    L = F.lib()
    assert (L.ffmi_debug_linear_tiles(T, N, K, epi | F.X_PACKED, None) == 10) == (K < 2560)  # (4120 x 2560: split)
    rng = np.random.default_rng(zlib.crc32(f"{T}:{N}:{K}".encode()))
    x = f16(rng.standard_normal((T, K)))
    W = [f16(rng.uniform(-0.05, 0.05, (N, K))) for _ in range(1 + epi)]
    dev = [Buf(w) for w in W]
    Wp = Buf.empty(((1 + epi) * L.ffmi_linear_packed_bytes(N, K) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_gate_up(dev[0].ptr, dev[1].ptr, N, K, Wp.ptr, None) if epi else
            L.ffmi_linear_pack_weight(dev[0].ptr, N, K, Wp.ptr, None))
    Xr, Xp = Buf(x), Buf(pack_act_np(x))
    y, z = (Buf(np.full((T + 1, N), np.nan, np.float16)) for _ in range(2))
    F.check(L.ffmi_linear(Xp.ptr, Wp.ptr, y.ptr, T, N, K, epi | F.X_PACKED | stream, None))
    F.check(L.ffmi_linear(Xr.ptr, Wp.ptr, z.ptr, T, N, K, epi | stream, None))
    y, z = y.get(), z.get()
    assert np.isnan(y[T]).all() and np.isfinite(y[:T]).all()
    assert np.array_equal(y[:T].view(np.uint16), z[:T].view(np.uint16))
    if not epi and T in (65, 192) and K < 512:
        close16(y[:T], O.linear(x.astype(np.float32), W[0].astype(np.float32), fp16=1))
