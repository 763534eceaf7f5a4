"""Picks without probabilities: rows whose maximum cannot tie are picked without their sum of
exponentials.  The same ids as the whole path gives, and as the oracle."""
import numpy as np
import pytest

import flexflow_amd.ffmi as F
import oracle_lib as O
from hip_util import Buf

pytestmark = pytest.mark.gpu


def rows(V, rng):
    out = [rng.standard_normal(V) * s for s in (1e-3, 0.02, 0.1, 1, 10, 300)]
    out += [np.zeros(V), np.full(V, -3.0)]  # flat: p is subnormal in long rows
    for top in (0.25, 0.9, 1.5, 3.0, 5.0, 40.0):  # one, two and eight fp16 steps below the maximum, ahead of it and behind
        for steps in (1, 2, 8):
            x = rng.standard_normal(V) * 0.05 - 2
            m = np.float16(top)
            below = np.float16(float(m) - steps * float(m - np.nextafter(m, np.float16(0))))
            at = rng.permutation(V)[:4]
            x[at[:2]], x[at[2:]] = m, below
            out.append(x)
    x = rng.standard_normal(V)
    x[rng.permutation(V)[:V // 2]] = -np.inf
    out.append(x)
    return np.stack(out).astype(np.float16)


@pytest.mark.parametrize("V", [8, 1000, 8192, 8200, 16400, 32000, 32768])
def test_picks(V):
    x = rows(V, np.random.default_rng(V))
    T, L = len(x), F.lib()
    lb, ids, both, pr = Buf(x), Buf.empty((T,), np.int32), Buf.empty((T,), np.int32), Buf.empty((T,), np.float32)
    F.check(L.ffmi_argmax(lb.ptr, T, V, ids.ptr, None, None))
    F.check(L.ffmi_argmax(lb.ptr, T, V, both.ptr, pr.ptr, None))
    assert ids.get().tolist() == both.get().tolist() == O.softmax_argmax(x.astype(np.float32), fp16=1)[0].tolist()


def test_rows_without_a_finite_maximum():
    x = np.random.default_rng(1).standard_normal((5, 1000)).astype(np.float16)
    x[0, 7] = np.nan
    x[1, :] = np.nan
    x[2, 5] = np.inf
    x[3, :] = -np.inf
    lb, ids, both, pr = Buf(x), Buf.empty((5,), np.int32), Buf.empty((5,), np.int32), Buf.empty((5,), np.float32)
    F.check(F.lib().ffmi_argmax(lb.ptr, 5, 1000, ids.ptr, None, None))
    F.check(F.lib().ffmi_argmax(lb.ptr, 5, 1000, both.ptr, pr.ptr, None))
    assert ids.get().tolist() == both.get().tolist()


# the forms of one to eight workgroups a row
@pytest.mark.parametrize("V", [1000, 8200, 32000])
@pytest.mark.parametrize("T", [1, 8, 33, 64, 65, 128, 129])
def test_rows_that_may_tie_share_their_sums(T, V):
    """Rows that need their sum of exponentials spread it over workgroups, as with probabilities (partial sums
    in the workspace, behind 1 KB of counters that are left zero); the others need none."""
    x, L = rows(V, np.random.default_rng(T)), F.lib()
    close, equal, clear = x[8], x[6], x[5]
    assert 0 < close.max() - np.unique(close)[-2] < 1e-3 and clear.max() - np.unique(clear)[-2] > 0.1
    n = int(L.ffmi_arg_topk_workspace_bytes(T))
    for row, sums in ((clear, False), (equal, False), (close, T <= 128 and V > 8192)):
        lb, ids, both = Buf(np.tile(row, (T, 1))), Buf.empty((T,), np.int32), Buf.empty((T,), np.int32)
        pr, ws, ws2 = Buf.empty((T,), np.float32), Buf(np.zeros(n, np.uint8)), Buf(np.zeros(n, np.uint8))
        F.check(L.ffmi_arg_topk_ws(lb.ptr, T, V, 1, ids.ptr, None, ws.ptr, n, None))
        F.check(L.ffmi_arg_topk_ws(lb.ptr, T, V, 1, both.ptr, pr.ptr, ws2.ptr, n, None))
        assert ids.get().tolist() == both.get().tolist()
        got, whole = ws.get(), ws2.get()
        assert not got[:1024].any() and not whole[:1024].any()
        assert got[1024:].any() == sums
        assert not sums or T == 1 or np.array_equal(got, whole)  # (one row takes two workgroups at most)
