"""Experts' lists: picked in their launch or in one before (up to 16 tokens at 64 columns and 16
picks, up to 8 otherwise), one, four and any number of picks a thread (1024, 4096)."""
import pytest

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
