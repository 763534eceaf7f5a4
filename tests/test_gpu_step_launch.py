"""Steps launched kernel by kernel and as graphs give the same bits, in turn on one model too."""
import numpy as np
import pytest

import flexflow_amd as fa
import flexflow_amd.ffmi as F

pytestmark = pytest.mark.gpu

CFG = dict(num_layers=2, vocab_size=500, num_heads=2, num_kv_heads=2, hidden=128, intermediate=256,
           rms_eps=1e-6, rope_theta=10000.0)


def replay(m, prompt, steps):
    rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_sequence_length=96)
    got = [rm.replay_step(m, [(1, prompt, range(len(prompt)))])]
    for k in range(steps):
        yield
        got.append(rm.replay_step(m, [(1, [7 + 3 * k], [0]), (2, [9 + k, 11], [1])]))
    yield np.concatenate(got)


@pytest.mark.parametrize("full", [False, True])
def test_same_bits(full, monkeypatch):
    prompt = [(37 * i) % 480 + 5 for i in range(20)]
    out = []
    for forms in ("1", "0", "10"):
        m = fa.Model(CFG, "inc", max_requests=2, max_tokens=64, max_seq_len=96, weight_seed=9, full_precision=full)
        for k, last in enumerate(replay(m, prompt, 12)):
            monkeypatch.setenv("FFMI_STEP_GRAPHS", forms[k % len(forms)])
        out.append(last)
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_same_tokens(monkeypatch):
    out = []
    for form in ("1", "0"):
        monkeypatch.setenv("FFMI_STEP_GRAPHS", form)
        m = fa.Model(CFG, "inc", max_requests=3, max_tokens=64, max_seq_len=96, weight_seed=9)
        rm = fa.RequestManager(max_requests_per_batch=3, max_tokens_per_batch=64, max_sequence_length=96)
        out.append([r.output_tokens for r in fa.generate(rm, m, [[5, 6, 7], [8, 9], [10]], max_length=60)])
    assert out[0] == out[1]


def test_form_by_counted_launches():
    """16 MB a launch, of as many launches as the step has: 24 with one token (norms in the products around
    them: 16.4 MB), 31 with 20 (12.7)."""
    cfg = dict(num_layers=4, vocab_size=8000, num_heads=16, num_kv_heads=16, hidden=2048, intermediate=4608,
               rms_eps=1e-6, rope_theta=10000.0)
    m = fa.Model(cfg, "inc", max_requests=1, max_tokens=64, max_seq_len=64, weight_seed=9)
    rm = fa.RequestManager(max_requests_per_batch=1, max_tokens_per_batch=64, max_sequence_length=64)
    for tokens, graphs in (([5], 0), (list(range(20)), 1), ([6], 1)):
        rm.replay_step(m, [(1, tokens, [0])])
        assert F.lib().ffmi_model_debug_graphs(m.handle) == graphs
