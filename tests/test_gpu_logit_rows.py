"""Logits of a replay step on their way to the host (runtime/logit_rows.h): more rows
than the staging's halves hold, any order and repeats of `want`, a vocabulary that is
no multiple of the kernel's vectors, against the same rows one step at a time."""
import numpy as np
import pytest

import flexflow_amd as fa
from vapipel_models import layer, model_config

pytestmark = pytest.mark.gpu

LLAMA = dict(num_layers=1, num_heads=2, num_kv_heads=2, hidden=128, intermediate=256, rms_eps=1e-6,
             rope_theta=10000.0)


@pytest.mark.parametrize("kind", ["fp16", "fp32", "paged"])
@pytest.mark.parametrize("vocab", [500, 1203, 33001])
def test_many_rows(kind, vocab):
    cfg = model_config(vocab, 96, 128, [layer(3, 24, 16, 40, 0.2, 160)]) if kind == "paged" else \
        dict(LLAMA, vocab_size=vocab)
    m = fa.Model(cfg, "inc", max_requests=2, max_tokens=64, max_seq_len=64, weight_seed=5,
                 full_precision=kind == "fp32")
    rm = fa.RequestManager(max_requests_per_batch=2, max_tokens_per_batch=64, max_spec_tree_token_num=0,
                           max_sequence_length=64)
    toks = [[(7 * i + 3 * r) % vocab for i in range(50)] for r in (0, 1)]
    whole = rm.replay_step(m, [(1, toks[0], range(50))])
    for want in ([49], range(16), range(17), range(33), [5, 3, 3, 41, 0], []):
        for rid in (2, 1):
            rm.replay_end(m, 1) if rid == 2 else None
            got = rm.replay_step(m, [(rid, toks[0], want)])
            rm.replay_end(m, rid) if rid == 2 else None
            assert got.shape == (len(want), vocab)
            assert np.array_equal(got, whole[list(want)])
    rm.replay_end(m, 1)
    # two requests in one step, the first one's rows out of order
    both = rm.replay_step(m, [(3, toks[0][:30], [29, 2]), (4, toks[1][:30], [1, 28])])
    assert both.shape == (4, vocab) and np.isfinite(both).all()
    assert np.abs(both[:2] - whole[[29, 2]]).max() < (1e-4 if kind == "fp32" else 3e-2) * np.abs(whole).max()
