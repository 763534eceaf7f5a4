"""Kernels of one workgroup per row take the rows in an order of their own (those of a packed line on one XCD): every
row once, whatever their number."""
import numpy as np
import pytest

import flexflow_amd.ffmi as F
import oracle_lib as O
from hip_util import Buf, f16, ulp_diff

pytestmark = pytest.mark.gpu


# fewer rows than XCDs, as many, one more, a remainder in every place, a prompt step's
@pytest.mark.parametrize("T", [1, 7, 8, 9, 15, 17, 64, 70, 185, 1023])
def test_residual_norm_rows(T):
    H, rng = 512, np.random.default_rng(T)
    x1, x2 = f16(rng.standard_normal((T, H))), f16(rng.standard_normal((T, H)))
    w = f16(rng.uniform(0.5, 1.5, H))
    r_ref, o_ref = O.residual_rmsnorm(x1.astype(np.float32), x2.astype(np.float32), w.astype(np.float32), 1e-6)
    a, b, wb = Buf(x1), Buf(x2), Buf(w)
    L = F.lib()
    tiles = (T + 15) // 16
    for flags, rows in ((0, T), (F.Y_PACKED, tiles * 16)):
        res, out = Buf(np.zeros((T, H), np.float16)), Buf(np.zeros((rows, H), np.float16))
        F.check(L.ffmi_rmsnorm_ex(a.ptr, b.ptr, wb.ptr, res.ptr, out.ptr, T, H, 1e-6, flags, None))
        got = out.get()
        if flags:  # tiles of 16 rows x 32 columns: [tile][k-block][8 columns of 4][row][8]
            got = got.reshape(tiles, H // 32, 4, 16, 8).transpose(0, 3, 1, 2, 4).reshape(rows, H)[:T]
        np.testing.assert_array_equal(res.get(), r_ref.astype(np.float16))
        assert ulp_diff(got, o_ref.astype(np.float16)).max() <= 1  # (the rms, a half, may round the other way)
