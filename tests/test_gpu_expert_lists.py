"""Experts: the router beside the norm that makes its rows; the lists, picked in their launch or in
one before (up to 16 tokens at 64 columns and 16 picks, up to 8 otherwise), of one, four and any
number of picks a thread (1024, 4096)."""
import numpy as np
import pytest

import flexflow_amd as fa

import nomutar_models as NM
import nomutar_ref as NR
import pekarax_models as PM
import pekarax_ref as PR
from test_gpu_nomutar import close as close_n, make_engine as engine_n, run as run_n, tokens as tokens_n
from test_gpu_pekarax import close as close_p, make_engine as engine_p, run as run_p, tokens as tokens_p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,top,T", [(64, 4, 16), (64, 4, 17), (65, 4, 8), (65, 4, 9), (32, 16, 64), (32, 16, 65),
                                     (40, 17, 8), (40, 17, 9), (24, 20, 204), (24, 20, 205)])
def test_lists(tmp_path, n, top, T):
    cfg = NM.model_config(90, 96, [NM.experts(NM.plain(2, 1, 16, 16, 0.2), n, top, 40, shared=70)], bigram=None)
    w = NM.random_weights(cfg, 7)
    toks = tokens_n(cfg, T, 5)
    eng = engine_n(NM.write_checkpoint(tmp_path / "n", cfg, w), False, pool=16 * 64, batch=256, positions=256)
    close_n(run_n(eng, toks, [T]), NR.forward(cfg, w, toks), False)
    cfg = PM.model_config(90, 96, [PM.experts(PM.gla(1, 16, 16), n - 4, top, 40, identity=4, groups=(1, 1))])
    w = PM.random_weights(cfg, 7)
    toks = tokens_p(cfg, T, 5)
    eng = engine_p(PM.write_checkpoint(tmp_path / "p", cfg, w), False, pool=16 * 64, batch=256, positions=256)
    close_p(run_p(eng, toks, [T]), PR.forward(cfg, w, toks), False)


@pytest.mark.parametrize("n,identity,width,T", [
    (12, 4, 96, 1), (12, 5, 100, 16), (30, 4, 352, 17), (47, 2, 1500, 16), (60, 4, 1536, 16), (60, 4, 1568, 16),
    (60, 4, 1568, 17), (61, 4, 96, 9), (33, 2, 4096, 64), (33, 2, 4096, 65), (33, 2, 4128, 20)])
def test_router_beside_the_norm(tmp_path, n, identity, width, T):
    """Up to 64 columns, 64 tokens and 4096 channels, with up to 16 tokens 6144 channels of 16
    columns; what lies past each."""
    cfg = PM.model_config(60, width, [PM.experts(PM.gla(1, 16, 16), n, 3, 32, identity=identity, groups=(1, 1))])
    w = PM.random_weights(cfg, 9)
    toks = tokens_p(cfg, T, 6)
    eng = engine_p(PM.write_checkpoint(tmp_path / "p", cfg, w), False, pool=16 * 64, batch=320, positions=320)
    close_p(run_p(eng, toks, [T]), PR.forward(cfg, w, toks), False)


@pytest.mark.parametrize("n,top,T,kinds", [
    (8, 2, 33, 90), (8, 2, 47, 90), (8, 2, 48, 90), (16, 4, 47, 90), (16, 4, 48, 90), (64, 1, 200, 90),
    (16, 4, 47, 2), (40, 4, 47, 1), (40, 1, 160, 1), (40, 1, 200, 2), (40, 2, 160, 6)])
def test_few_and_many_rows_an_expert(tmp_path, n, top, T, kinds):
    """Products of 16 rows a workgroup up to 4 rows an expert on average, up to 12 of up to 64 rows
    (tokens of few kinds: 17 to 64 rows of one expert, and more), from there on of 256."""
    cfg = PM.model_config(90, 96, [PM.experts(PM.gla(1, 16, 16), n, top, 200, identity=0, groups=(1, 1))])
    w = PM.random_weights(cfg, 11)
    toks = [t % kinds for t in tokens_p(cfg, T, 8)]
    eng = engine_p(PM.write_checkpoint(tmp_path / "p", cfg, w), False, pool=16 * 64, batch=256, positions=256)
    close_p(run_p(eng, toks, [T]), PR.forward(cfg, w, toks), False)


def many_requests(tmp_path, cfg):
    folder = PM.write_checkpoint(tmp_path / "p", cfg, PM.random_weights(cfg, 9))
    m = fa.Model(fa.load_config(folder), "inc", max_requests=64, max_tokens=64, max_seq_len=64, weights_folder=folder,
                 kv_pool_tokens=64 * 64)
    m.set_debug(True)
    return fa.RequestManager(max_requests_per_batch=64, max_tokens_per_batch=64, max_spec_tree_token_num=0,
                             max_sequence_length=64), m


def hidden(rm, m, toks, rid):
    """a step of requests of one token each: the residual stream after the first layer"""
    step = [(rid + i, [t], [0]) for i, t in enumerate(toks)]
    rm.replay_step(m, step)
    got = m.debug_tensor("hidden", 0)
    assert got.shape[0] == len(toks) and got.dtype == np.float32
    for e in step:
        rm.replay_end(m, e[0])
    return got


@pytest.mark.parametrize("n,identity,width", [(12, 4, 100), (40, 4, 544), (40, 4, 1024), (40, 4, 2048), (60, 4, 1568),
                                              (40, 4, 2080), (40, 4, 3104), (40, 4, 4096), (8, 4, 4096)])
def test_a_row_does_not_know_its_step(tmp_path, n, identity, width):
    """What a layer leaves of one token is the same bits in steps of 8 to 64 tokens, whose router is a product of
    its own or a part of the norm's launch: K whole, in slices, of k-steps that they do not divide."""
    cfg = PM.model_config(60, width, [PM.experts(PM.gla(1, 16, 16), n, 2, 32, identity=identity, groups=(1, 1))])
    rm, m = many_requests(tmp_path, cfg)
    # (up to 64 where the experts' products keep one order of sums)
    got = {T: hidden(rm, m, [(7 * i + 5) % 60 for i in range(T)], 100 * T)
           for T in ((8, 16, 17, 32, 64) if n >= 40 else (8, 16, 17, 32))}
    for T in got:
        assert np.array_equal(got[T][:16], got[17][:min(T, 16)]), T


@pytest.mark.parametrize("kinds", [60, 3, 1])
def test_some_and_many_rows_have_the_same_bits(tmp_path, kinds):
    """Experts' products of up to 64 rows a tile (33 and 59 tokens, 2 of 10 experts) and of 256 (60)."""
    cfg = PM.model_config(60, 544, [PM.experts(PM.gla(1, 16, 16), 10, 2, 328, identity=0, groups=(1, 1))])
    rm, m = many_requests(tmp_path, cfg)
    got = [hidden(rm, m, [(7 * i + 5) % kinds for i in range(T)], 100 * T) for T in (60, 59, 33)]
    for g in got:
        assert np.array_equal(g, got[0][:len(g)])
