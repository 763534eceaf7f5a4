"""Graphs of decode steps (llama_gpu.cpp attn_form): one per step shape where the
attention does not split a request's keys, one more for each number of workgroups that
share them where it does."""
import pytest

import flexflow_amd as fa
import flexflow_amd.ffmi as F

pytestmark = pytest.mark.gpu


def graphs_after(model, length):
    rm = fa.RequestManager(max_requests_per_batch=1, max_tokens_per_batch=64, max_spec_tree_token_num=0,
                           max_sequence_length=1200)
    res = fa.generate(rm, model, [[5, 17, 300]], max_length=length)
    assert len(res[0].output_tokens) == length
    return F.lib().ffmi_model_debug_graphs(model.handle)


# heads of 64 project in the attention's launch, which splits no keys; heads of 128 split
# them from 257 on (2 heads: 2 workgroups each, 3 from 513, 4 from 769, 5 from 1025)
@pytest.mark.parametrize("dim,more", [(64, [0, 0]), (128, [1, 3])])
def test_graphs_by_context(dim, more):
    cfg = dict(num_layers=1, vocab_size=1000, num_heads=2, num_kv_heads=2, hidden=2 * dim, intermediate=256,
               rms_eps=1e-6, rope_theta=10000.0)
    m = fa.Model(cfg, "inc", max_requests=1, max_tokens=64, max_seq_len=1200, weight_seed=3)
    short = graphs_after(m, 200)
    assert short > 0
    assert [graphs_after(m, n) - short for n in (400, 1000)] == more
