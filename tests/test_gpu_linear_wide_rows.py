"""Products of few rows: two column tiles a workgroup from 9 rows and 1536 tiles on; three row tiles.
A row's sums are the same bits however many rows there are."""
import numpy as np
import pytest

import flexflow_amd.ffmi as F
import test_gpu_kernels as K
from hip_util import Buf, f16

pytestmark = pytest.mark.gpu


def setup_module(module):
    K.setup_module(K)


@pytest.mark.parametrize("n,k,hint", [(24560, 1088, 0), (24576, 2048, F.W_STREAM), (24592, 1088, 0),
                                      (24600, 2048, F.W_STREAM), (32000, 1056, 0)])
def test_rows(n, k, hint):
    L = K.L
    rng = np.random.default_rng(n)
    x, w = f16(rng.standard_normal((17, k))), f16(rng.uniform(-0.05, 0.05, (n, k)))
    xb, wb, wp = Buf(x), Buf(w), Buf.empty((L.ffmi_linear_packed_bytes(n, k) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_weight(wb.ptr, n, k, wp.ptr, None))
    want = x.astype(np.float64) @ w.astype(np.float64).T
    # fp32 sums of k products (k 2^-24 of their magnitudes), rounded to fp16
    most = np.abs(x).astype(np.float32) @ np.abs(w).astype(np.float32).T
    bound = 2.0 ** -11 * np.abs(want) + k * 2.0 ** -24 * most + 2.0 ** -24
    got = {}
    for t in (16, 1, 8, 9, 12, 17):
        y = Buf(np.full((t, n), np.nan, np.float16))
        F.check(L.ffmi_linear(xb.ptr, wp.ptr, y.ptr, t, n, k, hint, None))
        got[t] = y.get()
        assert (np.abs(got[t].astype(np.float64) - want[:t]) <= bound[:t]).all(), t
        if t <= 16:
            assert np.array_equal(got[t].view(np.uint16), got[16][:t].view(np.uint16)), t


@pytest.mark.parametrize("n,k,epi,hint", [(6432, 2048, 0, F.W_STREAM), (2048, 4096, 0, 0), (2048, 1056, 0, 0),
                                          (768, 3072, 0, 0), (3072, 1536, 0, 0), (520, 2816, 0, 0), (8200, 1056, 0, 0), (2304, 768, 1, 0), (16400, 992, 0, 0)])
def test_rows_of_three_tiles(n, k, epi, hint):
    """33 to 48 rows have a form of their own; a row's sums are those of 64."""
    L = K.L
    rng = np.random.default_rng(n + k)
    x, w = f16(rng.standard_normal((64, k))), [Buf(f16(rng.uniform(-0.05, 0.05, (n, k)))) for _ in range(1 + epi)]
    xb, wp = Buf(x), Buf.empty(((1 + epi) * L.ffmi_linear_packed_bytes(n, k) // 2,), np.uint16)
    F.check(L.ffmi_linear_pack_gate_up(w[0].ptr, w[1].ptr, n, k, wp.ptr, None) if epi else
            L.ffmi_linear_pack_weight(w[0].ptr, n, k, wp.ptr, None))
    got = {}
    for t in (64, 32, 33, 40, 47, 48, 49):
        y = Buf(np.full((t, n), np.nan, np.float16))
        F.check(L.ffmi_linear(xb.ptr, wp.ptr, y.ptr, t, n, k, epi | hint, None))
        got[t] = y.get().view(np.uint16)
        assert np.array_equal(got[t], got[64][:t]), t
