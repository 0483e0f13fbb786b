"""Kernel variants at the sizes where they can go wrong: tile edges, remainders, the smallest and largest of the
range a dispatch rule gives them."""
import numpy as np
import pytest

import oracle
from helpers import mid_config, random_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from laya_amd.device import Context
    c = Context(0)
    yield c
    c.close()


def test_readout_option_counts(ctx):
    """The read-out keeps up to 256 options' exponentials in LDS and fetches the rest: one option, the last that
    fits, one past it, and more. Features of probabilities near 1/K: fp32 sums of K terms (K · 2^-24 ≈ 2e-5
    relative at most), held to 1e-5 absolute as the base-width read-out test does."""
    from laya_amd.batch import synthetic_batch
    from laya_amd.model import TrainableDecisionModel
    mc = mid_config(layers=1)
    o = oracle.OracleModel(mc, double=True)
    params = random_params(o.shapes, 5, std=0.05)
    batch = synthetic_batch(np.random.default_rng(6), [620, 520, 700, 12], [256, 257, 300, 1], [0, 1, 2, 0],
                            mc.encoder.vocab_size)
    o.set_params(params)
    o.forward(batch, training=False)
    probs_o, feats_o, _ = o.readout()
    m = TrainableDecisionModel(mc, ctx)
    m.set_params(params)
    m.forward(batch, training=False)
    _, probs, feats = m.readout()
    np.testing.assert_allclose(feats, feats_o, atol=1e-5)
    np.testing.assert_allclose(probs, probs_o, atol=1e-5)
    m.close()
