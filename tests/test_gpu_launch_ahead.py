"""Decoding steps launched ahead of the picks they continue give the tokens of steps run one by
one: requests that end by length and by token while others go on, more of them than slots."""
import numpy as np
import pytest

import flexflow_amd as fa
from flexflow_amd import ffmi as F

pytestmark = pytest.mark.gpu

CFG = dict(num_layers=2, vocab_size=500, num_heads=2, num_kv_heads=2, hidden=128, intermediate=256,
           rms_eps=1e-6, rope_theta=10000.0)


def ahead(m):
    return F.lib().ffmi_model_debug_count(m.handle, F.COUNT_AHEAD)


def tokens(slots, prompts, lengths, eos):
    """The tokens of two passes, and whether steps were launched ahead."""
    m = fa.Model(CFG, "inc", max_requests=slots, max_tokens=64, max_seq_len=96, weight_seed=9)
    out = []
    for _ in range(2):  # (on what the first pass left behind, too)
        rm = fa.RequestManager(max_requests_per_batch=slots, max_tokens_per_batch=64, max_sequence_length=96,
                               eos_token_ids=eos)
        guids = [rm.register_new_request(p, max_length=n) for p, n in zip(prompts, lengths)]
        rm.serve_incr_decoding(m)
        out.append([rm.get_generation_result(g).output_tokens for g in guids])
    return out, ahead(m) > 0


@pytest.mark.parametrize("slots,requests", [(1, 1), (1, 3), (4, 3), (4, 4), (4, 7), (20, 20)])
def test_same_tokens_as_one_by_one(slots, requests, monkeypatch):
    prompts = [[(37 * i + 11 * r) % 480 + 5 for i in range(3 + r % 5)] for r in range(requests)]
    lengths = [min(96, len(p) + (3, 40, 2, 17, 60)[r % 5]) for r, p in enumerate(prompts)]
    lengths[0] = 50
    monkeypatch.setenv("FFMI_INC_AHEAD", "0")
    (plain, _), taken = tokens(slots, prompts, lengths, [])
    assert not taken
    assert [len(t) for t in plain] == lengths
    # tokens that end some requests early, at different steps
    eos = sorted({t[len(t) - len(t) // 3] for t in plain[::2]})
    short, _ = tokens(slots, prompts, lengths, eos)
    assert short[0] == short[1] and any(len(a) < len(b) for a, b in zip(short[0], plain))
    monkeypatch.delenv("FFMI_INC_AHEAD")
    # (three requests by one slot: none while others wait, and the last has two tokens to come)
    assert tokens(slots, prompts, lengths, []) == ([plain, plain], (slots, requests) != (1, 3))
    assert tokens(slots, prompts, lengths, eos)[0] == short


def test_refuses_tokens_out_of_range_behind_steps_launched_ahead():
    m = fa.Model(CFG, "inc", max_requests=2, max_tokens=64, max_seq_len=96, weight_seed=9)
    for bad in (-1, 500):
        rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_sequence_length=96)
        assert len(fa.generate(rm, m, [[5, 6, 7]], max_length=30)[0].output_tokens) == 30
        with pytest.raises(F.FFMIError):
            rm.replay_step(m, [(1, [9, bad], [1])])


# (5 layers: many short launches, whose last part is a graph; 20 requests: norms of their own)
@pytest.mark.parametrize("requests,layers", [(1, 2), (4, 2), (1, 5), (4, 5), (20, 5), (20, 3)])
def test_no_step_for_nobody(requests, layers, monkeypatch):
    """A call that tokens end runs as many steps to their end as one by one: none for nobody."""
    prompts = [[(37 * i + 11 * r) % 480 + 5 for i in range(3 + r % 5)] for r in range(requests)]
    runs = []
    for mode in ("0", "1"):
        monkeypatch.setenv("FFMI_INC_AHEAD", mode)
        m = fa.Model(dict(CFG, num_layers=layers), "inc", max_requests=requests, max_tokens=64, max_seq_len=96,
                     weight_seed=9)

        def count(what):
            return F.lib().ffmi_model_debug_count(m.handle, what)

        def call(eos):
            rm = fa.RequestManager(max_requests_per_batch=requests, max_tokens_per_batch=64, max_sequence_length=96,
                                   eos_token_ids=eos)
            before = [count(F.COUNT_STEPS), ahead(m)]
            guids = [rm.register_new_request(p, max_length=60) for p in prompts]
            rm.serve_incr_decoding(m)
            return ([rm.get_generation_result(g).output_tokens for g in guids], count(F.COUNT_STEPS) - before[0],
                    ahead(m) - before[1])
        plain = call([])
        gen = [t[-(60 - len(p) - 1):] for t, p in zip(plain[0], prompts)]
        eos = sorted({max(set(g), key=g.index) for g in gen})  # (the latest to come first)
        runs.append([plain, call(eos), call([499]), call(eos)])
        assert all(len(t) < 60 for t in runs[-1][1][0])
        assert (plain[2] > 0) == (runs[-1][1][2] > 0) == (mode == "1")
    for one, two in zip(*runs):
        assert one[0] == two[0] and one[1] == two[1]


def test_row_without_a_pick(tmp_path, monkeypatch):
    """A row of NaN has no pick: the step after it is refused, launched ahead or not."""
    rng, H = np.random.default_rng(3), CFG["hidden"]
    st = {}
    for n, rows, cols in (("model.embed_tokens", 500, H), ("lm_head", 500, H)):
        st[n + ".weight"] = rng.uniform(-0.5, 0.5, (rows, cols)).astype(np.float32)
    for l in range(CFG["num_layers"]):
        p = f"model.layers.{l}."
        for n in ("input_layernorm", "post_attention_layernorm"):
            st[p + n + ".weight"] = np.ones(H, np.float32)
        for n, rows, cols in [("self_attn.%s_proj" % x, H, H) for x in "qkvo"] + \
                [("mlp.gate_proj", 256, H), ("mlp.up_proj", 256, H), ("mlp.down_proj", H, 256)]:
            st[p + n + ".weight"] = rng.uniform(-0.1, 0.1, (rows, cols)).astype(np.float32)
    st["model.norm.weight"] = np.ones(H, np.float32)

    def run(folder, eos):
        m = fa.Model(CFG, "inc", max_requests=2, max_tokens=64, max_seq_len=96, weights_folder=str(folder))
        rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_sequence_length=96,
                               eos_token_ids=eos)
        try:
            return [r.output_tokens for r in fa.generate(rm, m, [[5, 6, 7], [300, 9]], max_length=40)], ahead(m)
        except F.FFMIError:
            return None, ahead(m)
    fa.convert_hf_model(st, str(tmp_path / "a"))
    plain, _ = run(tmp_path / "a", [])
    gen = plain[0][-36:-8]  # (the latest to come first, with steps behind it)
    late = max(set(gen) - set(plain[1]) - {5, 6, 7}, key=gen.index)
    assert gen.index(late) > 3
    st["model.embed_tokens.weight"][late] = np.nan
    fa.convert_hf_model(st, str(tmp_path / "b"))
    for eos in ([], [499]):
        for mode in ("0", "1"):
            monkeypatch.setenv("FFMI_INC_AHEAD", mode)
            out, taken = run(tmp_path / "b", eos)
            assert out is None and (taken > 0) == (mode == "1")


def test_graphs_given_back_between_steps_launched_ahead():
    """A model keeps 512 step graphs; the shape after those gives them back while steps are on the stream."""
    prompts = [[5, 6, 7], [300, 9]]

    def graphs(m):
        return F.lib().ffmi_model_debug_graphs(m.handle)

    def generate(m):
        rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_sequence_length=96)
        before = ahead(m)
        out = [r.output_tokens for r in fa.generate(rm, m, prompts, max_length=80)]
        assert ahead(m) > before
        return out
    m = fa.Model(CFG, "inc", max_requests=2, max_tokens=64, max_seq_len=96, weight_seed=9)
    plain = generate(m)
    m.close()
    m = fa.Model(CFG, "inc", max_requests=2, max_tokens=64, max_seq_len=96, weight_seed=9)
    rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_sequence_length=96)
    for a in range(1, 64):
        for b in range(1, min(a, 64 - a) + 1):
            if graphs(m) < 511:  # (the prompts' step is the last before they are given back)
                rm.replay_step(m, [(1, range(a), range(a)), (2, range(b), range(b))])
                rm.replay_end(m, 1), rm.replay_end(m, 2)
    assert graphs(m) == 511
    assert generate(m) == plain
    assert 0 < graphs(m) < 20
    assert generate(m) == plain
