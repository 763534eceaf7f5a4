"""Full-precision products of packed weights: the rings of steps of up to 16 tokens (fewer
k-blocks a wave than the ring, as many, one and two more, several turns) against the tiles of
longer steps.  All forms add up an output in the same order, so logits are the same bit for bit."""
import numpy as np
import pytest

import flexflow_amd as fa

pytestmark = pytest.mark.gpu


# K = hidden for gate and up (packed at any width) and qkv, intermediate for down; from 1280 on
# the other products are packed too.  k-blocks of 32 over four waves: 1 .. 44 a wave
@pytest.mark.parametrize("hidden,heads,inter", [(32, 1, 64), (192, 3, 96), (544, 17, 160), (1024, 8, 1280),
                                                (1312, 41, 1376), (1280, 10, 2080), (2176, 17, 5632),
                                                (4224, 33, 1408)])
def test_steps_of_few_rows(hidden, heads, inter):
    cfg = dict(num_layers=1, vocab_size=1000, num_heads=heads, num_kv_heads=heads, hidden=hidden, intermediate=inter,
               rms_eps=1e-6, rope_theta=10000.0)
    m = fa.Model(cfg, "inc", max_requests=1, max_tokens=64, max_seq_len=64, weight_seed=7, full_precision=True)
    rm = fa.RequestManager(max_requests_per_batch=1, max_tokens_per_batch=64, max_spec_tree_token_num=0,
                           max_sequence_length=64)
    toks = [(37 * i + 5) % 1000 for i in range(40)]
    whole = rm.replay_step(m, [(1, toks, range(40))])
    rm.replay_end(m, 1)
    got, at = [], 0
    for n in (1, 9, 2, 16, 8, 4):
        got.append(rm.replay_step(m, [(1, toks[at:at + n], range(n))]))
        at += n
    rm.replay_end(m, 1)
    assert np.array_equal(np.concatenate(got).view(np.uint32), whole.view(np.uint32))
