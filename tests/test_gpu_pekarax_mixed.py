"""Matrix memories where a step has long portions and single tokens: short spans' steps in the
launch of the chunks (states of up to 128 rows, the gated rule's of up to 256, up to 256 workgroups)
and in one of their own."""
import pytest

import pekarax_models as PM
import pekarax_ref as R
from test_gpu_pekarax import close, make_engine, together, tokens

pytestmark = pytest.mark.gpu


def models(heads, dim, vdim):
    return PM.model_config(50, 48, [PM.delta(heads, heads // 2, dim, vdim, low=(9, 9)), PM.gla(heads, dim, vdim),
                                    PM.parallel((1, 1, 16, 16, 1.0), (heads, dim, vdim, 10.0), 0.3, 1.0)])


# heads, widths; steps of (tokens of each request)
@pytest.mark.parametrize("heads,dim,vdim", [(4, 32, 64), (2, 64, 33), (4, 128, 128), (2, 100, 200), (2, 256, 96),
                                            (2, 257, 40)])
def test_portions_beside_tokens(tmp_path, heads, dim, vdim):
    cfg = models(heads, dim, vdim)
    w = PM.random_weights(cfg, 8)
    rm, m = make_engine(PM.write_checkpoint(tmp_path / "m", cfg, w), False, batch=256)
    steps = [(20, 3, 0, 0), (17, 1, 0, 64), (65, 2, 1, 1), (1, 16, 130, 1), (1, 1, 1, 1)]
    seqs = [tokens(cfg, sum(s[i] for s in steps), 40 + i) for i in range(4)]
    for got, seq in zip(together(rm, m, seqs, steps), seqs):
        close(got, R.forward(cfg, w, seq), False)


@pytest.mark.parametrize("portion", [17 * 64, 17 * 64 + 1])
def test_most_workgroups(tmp_path, portion):
    """Delta rule, 12 heads, 4 spans: 17 chunks are 252 workgroups with the short spans', 18 are 264."""
    cfg = PM.model_config(50, 32, [PM.delta(12, 6, 32, 32)])
    w = PM.random_weights(cfg, 8)
    rm, m = make_engine(PM.write_checkpoint(tmp_path / "m", cfg, w), False, pool=24 * 64, batch=1200, positions=1200)
    steps = [(2, 3, 1, 0), (1, 1, 2, portion), (1, 1, 1, 1)]
    seqs = [tokens(cfg, sum(s[i] for s in steps), 40 + i) for i in range(4)]
    for got, seq in zip(together(rm, m, seqs, steps), seqs):
        close(got, R.forward(cfg, w, seq), False)
