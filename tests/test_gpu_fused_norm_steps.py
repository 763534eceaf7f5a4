"""Decode steps whose products norm their own operands (up to 16 tokens, 2048 to 4096 channels; the
residual in packed tiles, the norm weight in LDS) against steps with norm launches."""
import numpy as np
import pytest

import flexflow_amd as fa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,heads", [(2048, 16), (2112, 33), (4096, 32), (4160, 65)])
def test_steps(monkeypatch, hidden, heads):
    """Where the sum of squares is taken in another order, a row's rms may round the other way, and so may
    its products: 2^-11 of the values, twice for either norm of a layer."""
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
    assert np.abs(out[0] - out[1]).max() <= 8 * 2.0 ** -11 * np.abs(out[1]).max()
