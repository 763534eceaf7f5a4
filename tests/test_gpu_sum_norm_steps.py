"""Steps of one and two tokens of small models (up to 1024 channels), whose norms ride in the launch of the product
behind them, against steps with norm launches: the same bits."""
import numpy as np
import pytest

import flexflow_amd as fa
import flexflow_amd.ffmi as F

pytestmark = pytest.mark.gpu


# (hidden, heads, intermediate, vocab): one head's slab and one output tile of gate and up; 8, 12 and 16 slabs of the
# attention and of down; a width that is no power of two; heads of 32, whose o product leaves slabs of its own; an
# output product by waves with an odd tile and a ragged one
@pytest.mark.parametrize("hidden,heads,ff,vocab", [(64, 1, 32, 500), (512, 8, 288, 500), (768, 12, 3072, 32000),
                                                   (832, 13, 96, 1000), (1024, 16, 2048, 16403), (256, 8, 512, 777)])
def test_same_bits(monkeypatch, hidden, heads, ff, vocab):
    cfg = dict(num_layers=3, vocab_size=vocab, num_heads=heads, num_kv_heads=heads, hidden=hidden, intermediate=ff,
               rms_eps=1e-6, rope_theta=10000.0)
    seq = np.random.default_rng(5).integers(0, vocab, (2, 40)).tolist()
    out = []
    for mode in ("1", "0"):
        monkeypatch.setenv("FFMI_SUM_NORM", mode)
        m = fa.Model(cfg, "inc", max_requests=2, max_tokens=64, max_seq_len=64, weight_seed=11)
        rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_sequence_length=64)
        parts, at = [], [0, 0]

        def feed(*which):
            parts.append(rm.replay_step(m, [(r + 1, seq[r][at[r]:at[r] + k], range(k)) for r, k in which]))
            for r, k in which:
                at[r] += k
        feed((0, 9))
        for _ in range(2):  # (the second time from a captured step)
            feed((0, 1))
            feed((0, 2))
            feed((1, 1))
            feed((0, 1), (1, 1))
            feed((0, 2), (1, 1))  # three rows: norm launches, whichever buffer the residual was in
        out.append(np.concatenate(parts))
        assert (F.lib().ffmi_model_debug_count(m.handle, F.COUNT_MADE_NORMS) > 0) == (mode == "1")
        m.close()
    assert np.isfinite(out[0]).all() and np.ptp(out[0]) > 0
    assert np.array_equal(out[0], out[1])
