"""Logits of a replay step on their way to the host (runtime/logit_rows.h): more rows
than the staging's halves hold, any order and repeats of `want`, a vocabulary that is
no multiple of the kernel's vectors, against the same rows one step at a time."""
import os
import subprocess
import sys
import time

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


WAITS = """
import time
import numpy as np
import flexflow_amd as fa
from vapipel_models import layer, model_config
fa.set_device(0)  # (applies FFMI_SYNC)
LLAMA = dict(num_layers=8, num_heads=16, num_kv_heads=16, hidden=2048, intermediate=5632, rms_eps=1e-6,
             rope_theta=10000.0, vocab_size=2000)
cfg = model_config(2000, 2048, 1024, [layer(16, 128, 128, 256, 0.1, 5632)] * 8) if KIND == "paged" else LLAMA
m = fa.Model(cfg, "inc", max_requests=1, max_tokens=1000, max_seq_len=1024, weight_seed=5,
             full_precision=KIND == "fp32")
rm = fa.RequestManager(max_requests_per_batch=1, max_tokens_per_batch=1000, max_spec_tree_token_num=0,
                       max_sequence_length=1024)
toks = np.arange(1000, dtype=np.int32)
wall = cpu = 0.0
for i in range(24):
    w, c = time.perf_counter(), time.thread_time()
    rm.replay_step(m, [(i + 1, toks, [999])])
    if i >= 4:
        wall, cpu = wall + time.perf_counter() - w, cpu + time.thread_time() - c
    rm.replay_end(m, i + 1)
print("share", cpu / wall, wall / 20)
"""


@pytest.mark.parametrize("kind", ["fp16", "fp32", "paged"])
def test_a_long_step_is_waited_for_as_asked(kind):
    """FFMI_SYNC=block: the thread sleeps while a step of milliseconds runs (launching it is what is left)."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, FFMI_SYNC="block", PYTHONPATH=os.pathsep.join([root, os.path.join(root, "tests")]))
    r = subprocess.run([sys.executable, "-c", "KIND = %r\n" % kind + WAITS], env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    print(r.stdout)
    assert "not applied" not in r.stderr and float(r.stdout.split("share")[1].split()[0]) < 0.75, r.stdout


def fastest(vocab, rows, times=25):
    m = fa.Model(dict(LLAMA, vocab_size=vocab), "inc", max_requests=1, max_tokens=256, max_seq_len=256, weight_seed=5)
    rm = fa.RequestManager(max_requests_per_batch=1, max_tokens_per_batch=256, max_spec_tree_token_num=0,
                           max_sequence_length=256)
    best, toks = 1e9, np.arange(max(rows, 4), dtype=np.int32)
    for i in range(times):
        t = time.perf_counter()
        rm.replay_step(m, [(i + 1, toks, range(rows))])
        best = min(best, time.perf_counter() - t)
        rm.replay_end(m, i + 1)
    return best


def test_odd_and_short_rows_arrive_as_fast():
    """Rows that are no whole pieces of 16 bytes, and short ones, which lie in one workgroup: 48 rows of
    33001 take as long as of 33000 (3 times so in single words), 200 of 1000 less than five steps of
    one row (6.5 one after the other)."""
    odd, even = fastest(33001, 48), fastest(33000, 48)
    one, many = fastest(1000, 1), fastest(1000, 200)
    print("us", *(round(t * 1e6) for t in (odd, even, one, many)))
    assert odd < 1.6 * even and many < 5 * one
