"""Convolved rows (kernels/conv_rows.hip) with one, two and four tokens a thread: up to 640 Ki
elements (53 tokens of 12288 columns), up to 5 Mi (426), and more.  Portions that start at every
place of a thread's tokens, shorter than the taps and long, from carried rows and from none; the
oldest tap stands out, so that the row it reads decides."""
import numpy as np
import pytest

import flexflow_amd as fa
import pekarax_models as PM
import pekarax_ref as R
from test_gpu_pekarax import close, together, tokens

pytestmark = pytest.mark.gpu

HEADS, DIM = 64, 64  # queries, keys and values: 12288 columns
FIRST = (17, 17, 18, 50, 22, 2, 5, 23, 3, 31, 33, 1, 21, 1, 19, 19, 18, 27, 40, 25, 26, 30)
THEN = (21, 23, 19, 17, 18, 1, 2, 19, 1, 1, 22, 27, 18, 50, 40, 30, 31, 33, 27, 3, 26, 17)
FEW = (1, 17, 2, 0, 1, 3, 18, 1, 0, 4, 33, 1, 0, 0, 19, 0, 2, 0, 1, 0, 20, 5)
LEAST = (0, 18, 0, 1, 0, 2, 0, 0, 1, 0, 0, 3, 0, 17, 0, 1, 0, 0, 2, 0, 5, 1)


def test_the_steps_take_every_form():
    assert sum(FIRST) % 4 == 0 and sum(THEN) % 4  # whole groups of four, and a rest
    assert [n * 3 * HEADS * DIM for n in (53, 54, 426, 427)] == [651264, 663552, 5234688, 5246976]
    assert min(sum(FIRST), sum(THEN)) > 426 and 53 < sum(FEW) < 427 and sum(LEAST) < 54
    for step in (FIRST, THEN):
        starts = np.cumsum((0,) + step[:-1])
        for short in (True, False):
            assert {s % 4 for s, n in zip(starts, step) if (n < 4) == short} == {0, 1, 2, 3}


@pytest.mark.parametrize("taps,full", [(1, False), (2, False), (3, False), (4, False), (6, False), (2, True), (4, True),
                                       (6, True)])
def test_tokens_a_thread(tmp_path, taps, full):
    att = PM.parallel((HEADS, HEADS, DIM, DIM, 1.0, DIM, 100.0, taps), (1, 16, 16, 5.0), 1.0, 0.2)
    # (full precision convolves the delta rule's rows in the memory's launch)
    cfg = PM.model_config(64, 64, [att] if full else [att, PM.delta(HEADS, HEADS, DIM, DIM, conv=taps)])
    w = PM.random_weights(cfg, 4)
    for n in w:
        if n.endswith("conv") and taps > 1:
            w[n][:, 0] = 3.0
    folder, B = PM.write_checkpoint(tmp_path / "c", cfg, w), len(FIRST)
    m = fa.Model(fa.load_config(folder), "inc", max_requests=B, max_tokens=512, max_seq_len=192, weights_folder=folder,
                 full_precision=full, kv_pool_tokens=3 * 64 * B)
    rm = fa.RequestManager(max_requests_per_batch=B, max_tokens_per_batch=512, max_spec_tree_token_num=0,
                           max_sequence_length=192)
    steps = (FIRST, THEN, FEW, LEAST)
    seqs = [tokens(cfg, sum(s[i] for s in steps), 60 + i) for i in range(B)]
    got = together(rm, m, seqs, steps)
    close(np.concatenate(got), np.concatenate([R.forward(cfg, w, s) for s in seqs]), full)
    rows = np.array([len(g) for g in got])
    if not full and taps > 1:  # (a planted mistake must be seen: the taps in the other order)
        turned = {n: a[:, ::-1] if n.endswith("conv") else a for n, a in w.items()}
        with pytest.raises(AssertionError):
            close(np.concatenate(got), np.concatenate([R.forward(cfg, turned, s) for s in seqs]), full)
    assert rows.sum() == sum(map(sum, steps))
