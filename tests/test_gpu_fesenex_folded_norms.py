"""Steps without norm launches (up to 16 tokens, 2048 to 4096 channels): the product before a norm
leaves x w and its squares, the one after it scales its sums.  Layers with and without a
feed-forward, of either mixer; channels that are no multiple of 32."""
import pytest

import fesenex_models as FM
import fesenex_ref as R
from test_gpu_fesenex import close, make_engine, run, tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [2010, 2017, 2048, 2500, 4090, 4100])
def test_steps(tmp_path, width):
    model = FM.model_config(80, width, [FM.attention(2, 1, 32, 32, 0.2, ff=96), FM.lightning(2, 32, 32, [0.9, 0.8]),
                                        FM.attention(2, 2, 64, 32, 0.2), FM.lightning(1, 32, 64, [0.95], ff=64)])
    weights = FM.random_weights(model, 4)
    eng = make_engine(FM.write_checkpoint(tmp_path / "m", model[0], weights), False)
    toks = tokens(model, 60, width)
    close(run(eng, toks, [3, 1, 15, 16, 17, 1, 7]), R.forward(model[0], weights, toks, []), False)


@pytest.mark.parametrize("width,ff", [(2048, 8192), (2048, 8200), (2080, 8200)])
def test_long_products(tmp_path, width, ff):
    """The second product of a feed-forward in two slices of K, beside a norm of its own, beyond
    8192 units of 2048 channels; the mixer's stays as it is."""
    model = FM.model_config(80, width, [FM.attention(2, 1, 32, 32, 0.2, ff=ff), FM.lightning(2, 32, 32, [0.9, 0.8]),
                                        FM.lightning(1, 32, 64, [0.95], ff=64)])
    weights = FM.random_weights(model, 4)
    eng = make_engine(FM.write_checkpoint(tmp_path / "m", model[0], weights), False)
    toks = tokens(model, 40, width)
    close(run(eng, toks, [3, 1, 16, 17, 1, 2]), R.forward(model[0], weights, toks, []), False)
