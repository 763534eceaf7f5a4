"""Long steps of the LLaMA models whose callers read few rows: the final norm, lm_head and
sampling run on those rows only.  Logits against the same step with every row computed
(debug capture), tokens of prompts of that kind against prompts in short portions.  In full
precision every form of a product adds up in the same order, so there a token's logits do
not depend on its step at all."""
import numpy as np
import pytest

import flexflow_amd as fa

pytestmark = pytest.mark.gpu

CFG = dict(num_layers=2, vocab_size=500, num_heads=2, num_kv_heads=2, hidden=128, intermediate=256,
           rms_eps=1e-6, rope_theta=10000.0)


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("T", [64, 65, 66, 130, 256, 300])
def test_rows_of_a_long_step(T, full):
    m = fa.Model(CFG, "inc", max_requests=3, max_tokens=256, max_seq_len=320, weight_seed=7, full_precision=full)
    rm = fa.RequestManager(max_requests_per_batch=3, max_tokens_per_batch=256, max_sequence_length=320)
    rng = np.random.default_rng(T)
    n = [T - 11, 10, 1]
    toks = [rng.integers(3, 500, k).astype(np.int32) for k in n]

    def step(want):
        got = rm.replay_step(m, [(r + 1, t, w) for r, (t, w) in enumerate(zip(toks, want))])
        more = rm.replay_step(m, [(2, [77], [0])])  # (and what the step left behind is whole)
        for r in range(3):
            rm.replay_end(m, r + 1)
        return np.concatenate([got, more])
    every = step([range(n[0]), range(10), [0]])  # (every row is wanted, so every row is computed)
    for want in ([[n[0] - 1], [9], [0]], [[], [], [0]], [[], [], []], [list(range(0, n[0], 3)), [4, 2], []],
                 [list(range(max(0, T // 2 - 2))), [0], []], [range(n[0]), range(10), [0]]):
        few = step(want)
        m.set_debug(True)  # (every row)
        whole = step(want)
        m.set_debug(False)
        assert few.shape == whole.shape == (sum(map(len, want)) + 1, 500)
        # 16 bits: the logits are rounded to half (2^-11 of a value) after sums of 128 products in another order
        # (less than that), and lm_head's inputs are the same; 32 bits: sums of 128 products, 128 * 2^-24 of |x||w|
        bound = (2.0 ** -10 * np.abs(whole) + 2.0 ** -14 * np.abs(whole).max()) if not full else 1e-5 * np.abs(whole).max()
        assert (np.abs(few[:-1] - whole[:-1]) <= bound[:-1] if not full else
                np.abs(few[:-1] - whole[:-1]) <= bound).all()
        # a step after it: the long step's own keys and values, whatever rows it was asked for, are the same
        # bits; those of a step under debug capture (other kernels in 16 bits) are as near as 16 bits are
        assert np.array_equal(few[-1], every[-1])
        assert np.abs(few[-1] - whole[-1]).max() <= (2e-2 if not full else 1e-5) * np.abs(whole).max()


@pytest.mark.parametrize("full", [False, True])
def test_prompts_together_and_in_portions(full):
    out = []
    for step in (256, 40):  # tokens of a step: every prompt at once, or in portions that take every row
        m = fa.Model(CFG, "inc", max_requests=3, max_tokens=256, max_seq_len=320, weight_seed=3,
                     weight_init="token_chain", full_precision=full)
        rm = fa.RequestManager(max_requests_per_batch=3, max_tokens_per_batch=step, max_sequence_length=320)
        prompts = [[(31 * i + 7 * r) % 490 + 5 for i in range(k)] for r, k in enumerate((150, 33, 60))]
        out.append([r.output_tokens for r in fa.generate(rm, m, prompts, max_new_tokens=8)])
    assert out[0] == out[1]


# widths that meet half tiles of columns, whole ones, rings of two and four k-blocks, gate and up columns in one
# tile, widths that are no multiple of 8 (up to 16 tokens), and the forms of more tokens
@pytest.mark.parametrize("ff,vocab", [(256, 500), (2080, 2101), (4128, 4101)])
def test_full_precision_does_not_depend_on_the_step(ff, vocab):
    m = fa.Model(dict(CFG, intermediate=ff, vocab_size=vocab), "inc", max_requests=1, max_tokens=128, max_seq_len=128,
                 weight_seed=9, full_precision=True)
    rm = fa.RequestManager(max_requests_per_batch=1, max_tokens_per_batch=128, max_sequence_length=128)
    toks = [(37 * i + 11) % vocab for i in range(90)]
    whole = rm.replay_step(m, [(1, toks, range(90))])
    rm.replay_end(m, 1)
    got, at = [], 0
    for k in (1, 2, 8, 9, 16, 17, 7, 1, 29):
        got.append(rm.replay_step(m, [(1, toks[at:at + k], range(k))]))
        at += k
    rm.replay_end(m, 1)
    assert at == 90 and np.array_equal(np.concatenate(got), whole) and np.isfinite(whole).all() and whole.std() > 0


# the same at widths of which every weight is kept in blocks: half tiles of columns (heads, ff), whole ones in
# rings of two and of four k-blocks (qkv and lm_head), pairs, columns past the last whole tile, and numbers of
# columns that the workgroups of an XCD take in one piece
@pytest.mark.parametrize("hidden,ff,vocab", [(1280, 1312, 2101), (1280, 2080, 4101), (1536, 1280, 4097),
                                             (1280, 2048, 4096), (2048, 1280, 6144)])
def test_full_precision_of_wide_rows_does_not_depend_on_the_step(hidden, ff, vocab, monkeypatch):
    monkeypatch.setitem(CFG, "hidden", hidden)
    monkeypatch.setitem(CFG, "num_heads", hidden // 128)
    monkeypatch.setitem(CFG, "num_kv_heads", hidden // 128)
    test_full_precision_does_not_depend_on_the_step(ff, vocab)
