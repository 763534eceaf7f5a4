"""Steps launched kernel by kernel and as graphs give the same bits, in turn on one model too."""
import numpy as np
import pytest

import fesenex_models
import flexflow_amd as fa
import flexflow_amd.ffmi as F
import nomutar_models
import pekarax_models
import vapipel_models

pytestmark = pytest.mark.gpu

CFG = dict(num_layers=2, vocab_size=500, num_heads=2, num_kv_heads=2, hidden=128, intermediate=256,
           rms_eps=1e-6, rope_theta=10000.0)


def graphs(m):
    return F.lib().ffmi_model_debug_graphs(m.handle)


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
        monkeypatch.setenv("FFMI_STEP_GRAPHS", forms[0])
        m = fa.Model(CFG, "inc", max_requests=2, max_tokens=64, max_seq_len=96, weight_seed=9, full_precision=full)
        for k, last in enumerate(replay(m, prompt, 12)):
            monkeypatch.setenv("FFMI_STEP_GRAPHS", forms[k % len(forms)])
        out.append(last)
        assert (graphs(m) > 0) == ("1" in forms)
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_same_tokens(monkeypatch):
    out = []
    for form in ("1", "0"):
        monkeypatch.setenv("FFMI_STEP_GRAPHS", form)
        m = fa.Model(CFG, "inc", max_requests=3, max_tokens=64, max_seq_len=96, weight_seed=9)
        rm = fa.RequestManager(max_requests_per_batch=3, max_tokens_per_batch=64, max_sequence_length=96)
        out.append([r.output_tokens for r in fa.generate(rm, m, [[5, 6, 7], [8, 9], [10]], max_length=60)])
        assert (graphs(m) > 0) == (form == "1")
    assert out[0] == out[1]


def test_form_by_counted_launches():
    """14 MB a launch, of as many launches as the step has: 24 with one token (norms in the products around
    them: 16.4 MB), 31 with 20 (12.7)."""
    cfg = dict(num_layers=4, vocab_size=8000, num_heads=16, num_kv_heads=16, hidden=2048, intermediate=4608,
               rms_eps=1e-6, rope_theta=10000.0)
    m = fa.Model(cfg, "inc", max_requests=1, max_tokens=64, max_seq_len=64, weight_seed=9)
    rm = fa.RequestManager(max_requests_per_batch=1, max_tokens_per_batch=64, max_sequence_length=64)
    for tokens, held in (([5], 0), (list(range(20)), 1), ([6], 1)):
        rm.replay_step(m, [(1, tokens, [0])])
        assert graphs(m) == held


def paged(family):
    if family == "vapipel":
        v = vapipel_models
        return v.model_config(300, 128, 96, [v.layer(4, 32, 32, 64, 0.2, 256), v.layer(4, 32, 32, 64, 0.2, None)])
    if family == "fesenex":
        f = fesenex_models
        return f.model_config(300, 128, [f.attention(4, 2, 32, 32, 0.2, ff=256), f.lightning(4, 32, 32, [0.5, 0.7, 0.9, 1])])[0]
    if family == "nomutar":
        n = nomutar_models
        return n.model_config(300, 128, [n.dense(n.turned(4, 2, 32, 32, 0.2), 256),
                                         n.experts(n.plain(4, 2, 32, 32, 0.2), 8, 2, 64, 64)], cap=20.0)
    p = pekarax_models
    return p.model_config(300, 128, [p.experts(p.parallel((4, 2, 32, 32, 0.2), (2, 32, 32, 10.0)), 8, 2, 64),
                                     p.delta(2, 2, 32, 32), p.experts(p.gla(2, 32, 32), 8, 2, 64, identity=2)])


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("family", ["vapipel", "fesenex", "nomutar", "pekarax"])
def test_paged_families_same_bits(family, full, monkeypatch):
    prompt = [(37 * i) % 280 + 5 for i in range(40)]
    out = []
    for forms in ("1", "0", "10"):
        monkeypatch.setenv("FFMI_STEP_GRAPHS", forms[0])
        m = fa.Model(paged(family), "inc", max_requests=2, max_tokens=64, max_seq_len=96, weight_seed=9,
                     full_precision=full)
        for k, last in enumerate(replay(m, prompt, 12)):
            monkeypatch.setenv("FFMI_STEP_GRAPHS", forms[k % len(forms)])
        out.append(last)
        assert (graphs(m) > 0) == ("1" in forms)
    assert np.isfinite(out[0]).all() and np.ptp(out[0]) > 0
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_captured_but_launched_one_by_one(monkeypatch):
    """A step whose graph is not kept, as its capture has few launches: 311 MB, 15 of them."""
    f = fesenex_models
    cfg = f.model_config(32000, 2048, [f.attention(16, 4, 128, 128, 0.09, ff=5632)] * 2)[0]
    out = []
    for form in (None, "1"):
        if form:
            monkeypatch.setenv("FFMI_STEP_GRAPHS", form)
        m = fa.Model(cfg, "inc", max_requests=2, max_tokens=64, max_seq_len=96, weight_seed=9)
        *_, last = replay(m, list(range(5, 25)), 4)
        out.append(last)
        assert (graphs(m) > 0) == (form == "1")
        m.close()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])
