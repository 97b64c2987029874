"""Predictions on both sides of the batch size from which one thread takes a
whole sample (kManySamples, exachem_amd/csrc/xt_mlp.hip)."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from test_cost_model import rand_params


@pytest.mark.gpu
@pytest.mark.parametrize("n", [32767, 32768, 32769, 33023])
def test_predictions_of_both_forms_are_the_same_bits(xt, n):
    """Both sum in the same order, so a batch equals its parts bit for bit; the
    tolerance against the oracle is that of test_mlp_batches."""
    m = xt.CostModel(0, seed=1)
    p = rand_params(7).astype(np.float32)
    m.set_params(p)
    x = np.random.default_rng(n).uniform(-1.0, 1.0, (n, 7)).astype(np.float32)
    y = m.predict(x)
    half = n // 2
    assert np.array_equal(y, np.concatenate([m.predict(x[:half]), m.predict(x[half:])]))
    ref = MO.forward(p.astype(np.float64), x.astype(np.float64))[0]
    assert np.max(np.abs(y - ref)) <= 1e-5 * max(1.0, np.max(np.abs(ref)))
    m.close()
