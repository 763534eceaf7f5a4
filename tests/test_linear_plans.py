"""Which kernel takes a dense layer's product (gemm_kernels.h tile_plan, msplit_ahead), on
the CPU: the plan is host code."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import pytest

import flexflow_amd.ffmi as F


def tiles(T, N, K, epi=0):
    """(form, slices) of the tile kernel, None where another kernel takes the product"""
    s = ctypes.c_int()
    form = F.lib().ffmi_debug_linear_tiles(T, N, K, epi, ctypes.byref(s))
    return (form, s.value) if form >= 0 else None


# two blocks of up to 192 rows: short slices of packed activations stay with the M-split kernel
@pytest.mark.parametrize("T", [257, 300, 352, 384])
@pytest.mark.parametrize("N,K,epi,ours", [
    (2304, 768, 0, True), (2048, 512, 0, True), (8192, 1024, 0, True), (1024, 256, 0, True), (2816, 1024, 1, True),
    (512, 4096, 0, True), (256, 2048, 0, True), (128, 2048, 0, True), (64, 4096, 0, True),
    (768, 768, 0, False), (768, 3072, 0, False), (1024, 1024, 0, False), (32000, 768, 0, False),
    (2304, 2048, 0, False), (6144, 2048, 0, False), (4096, 2048, 0, False), (128, 512, 0, False)])
def test_two_row_blocks(T, N, K, epi, ours):
    assert (tiles(T, N, K, epi | F.X_PACKED) is None) == ours
    assert tiles(T, N, K, epi) is not None


@pytest.mark.parametrize("flags", [0, F.X_PACKED])
@pytest.mark.parametrize("T,N,K,epi,ours", [(257, 12288, 4096, 0, True), (384, 4096, 11008, 0, True),
                                            (384, 11008, 4096, 1, False), (385, 12288, 4096, 0, False)])
def test_large_weights(T, N, K, epi, ours, flags):
    assert (tiles(T, N, K, epi | flags) is None) == ours


# row-major activations are packed first: workspace for more than the slabs
@pytest.mark.parametrize("T,N,K,epi,packs", [
    (257, 2048, 2048, 0, True), (300, 4096, 2048, 0, True), (257, 1024, 1024, 0, True), (193, 768, 768, 0, True),
    (1024, 768, 768, 0, False), (300, 512, 4096, 0, False), (300, 4096, 1376, 0, False), (300, 2304, 768, 0, False),
    (192, 2048, 2048, 0, False), (168, 12288, 4096, 0, True), (128, 12288, 4096, 0, False)])
def test_packed_first(T, N, K, epi, packs):
    L = F.lib()
    slabs = L.ffmi_linear_workspace_bytes(T, N, K, epi | F.X_PACKED)
    both = (slabs + 255) // 256 * 256 + L.ffmi_packed_activation_bytes(T, K)
    assert L.ffmi_linear_workspace_bytes(T, N, K, epi) == (both if packs else slabs)


@pytest.mark.parametrize("T", [1, 64, 65, 192, 193, 256, 385, 1024])
def test_row_range(T):
    assert (tiles(T, 2304, 768) is not None) == (T > 192)


@pytest.mark.parametrize("N,K", [(2304, 768), (512, 2048), (4096, 4096), (1536, 4096)])
def test_row_tiles_alone_decide(N, K):
    """A thread keeps its plans by row tiles: they must not depend on which T asked first."""
    def asked(first):
        with ThreadPoolExecutor(1) as one:  # (a thread that has kept none)
            return one.submit(lambda: [tiles(16 * t + first, N, K, F.X_PACKED) for t in range(12, 30)]).result()
    assert all(asked(r) == asked(16) for r in range(1, 16))


@pytest.mark.parametrize("epi", [0, 1])
def test_every_tile_form_is_tested(epi, monkeypatch):
    """test_gpu_tile_gemm.py meets every form, in and out of K slices."""
    import test_gpu_tile_gemm as G
    monkeypatch.setenv("FFMI_TILE_GEMM", "2")
    met = {(form, sliced) for _, _, _, e, form, sliced in G.FORMS if e == epi}
    for T, N, K in G.CASES:
        N = N // 2 if epi and N > 8000 else N
        form, slices = tiles(T, N + (-N % 32 if epi else 0), K, epi)
        met.add((form, slices > 1))
    assert met == {(form, sliced) for form in range(10) for sliced in (False, True)}
    for T, N, K, e, form, sliced in G.FORMS:
        got = tiles(T, N, K, e)
        assert (got[0], got[1] > 1) == (form, sliced)


# up to 64 rows a call of its own never splits K: nothing to keep
@pytest.mark.parametrize("T", [1, 16, 64])
@pytest.mark.parametrize("N,K", [(768, 768), (2048, 2048), (6144, 2048), (12320, 4096), (32000, 768)])
def test_few_rows_need_no_workspace(T, N, K):
    assert F.lib().ffmi_linear_workspace_bytes(T, N, K, 0) == 0


# halves of K only where the grid that runs gains by them: one tile of 16 columns a workgroup, two from 512
# tiles and 17 rows on; whole K where a wave takes it; the same for every T
@pytest.mark.parametrize("N,K,slices", [
    (2048, 2048, 2), (2048, 1376, 2), (6144, 4096, 2), (4608, 4096, 2), (5632, 2048, 2), (9600, 4096, 2),
    (8224, 2048, 2), (4096, 4096, 1), (4096, 11008, 1), (12288, 4096, 1), (12320, 2048, 1), (12576, 4096, 1),
    (22016, 4096, 1), (22016, 1024, 1), (16448, 1024, 1), (16448, 1056, 2), (32000, 4096, 1), (2048, 992, 1)])
def test_halves_of_few_rows(N, K, slices):
    L = F.lib()
    assert {L.ffmi_debug_few_rows_slices(T, N, K) for T in (1, 16, 17, 33, 64)} == {slices}


# 65 .. 192 rows of packed activations, 96 columns a workgroup, whole K: twelve waves, unless the tile kernel
# is off; what is split in K stays with the M-split kernel
@pytest.mark.parametrize("T", [65, 128, 129, 192])
@pytest.mark.parametrize("N,K,epi,ours", [(11008, 4096, 1, True), (20480, 4096, 0, True), (18432, 512, 0, True),
                                          (12288, 4096, 0, False), (6144, 2048, 0, False), (6144, 4096, 0, False),
                                          (5632, 4096, 1, False), (32000, 4096, 0, False), (4096, 4096, 0, False)])
def test_twelve_waves(T, N, K, epi, ours, monkeypatch):
    assert tiles(T, N, K, epi | F.X_PACKED) == ((10, 1) if ours else None)
    assert tiles(T, N, K, epi) is None
    monkeypatch.setenv("FFMI_TILE_GEMM", "0")
    assert tiles(T, N, K, epi | F.X_PACKED) is None
