"""Cost model kernels at the edges of their sample chunks and of the captured
replay: loss, gradient and a few training steps against the CPU checker."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from test_cost_model import batch, rand_params


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 129, 4097])
def test_gradient_and_forward_at_chunk_edges(xt, n):
    """Tolerance: sums of up to n + 64 FP32 terms, each within 2^-24 of its
    value; 1e-5 of the largest entry covers n = 4097 with random signs."""
    m = xt.CostModel(0, seed=1)
    p = rand_params(21).astype(np.float32)
    m.set_params(p)
    x, t = (v.astype(np.float32) for v in batch(22, n))
    loss, g = m.loss_grad(x, t)
    p64, x64, t64 = p.astype(np.float64), x.astype(np.float64), t.astype(np.float64)
    rl, rg = MO.loss_grad(p64, x64, t64)
    assert abs(loss - rl) <= 1e-5 * abs(rl) + 1e-7
    assert np.max(np.abs(g - rg)) <= 1e-5 * np.max(np.abs(rg)) + 1e-7
    y = MO.forward(p64, x64)[0]
    assert np.max(np.abs(m.predict(x) - y)) <= 1e-5 * max(1.0, np.max(np.abs(y)))
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 31, 63, 64, 65, 97])
def test_replayed_and_direct_steps_agree(xt, steps):
    """A call of `steps` steps (captured blocks and the rest launched) gives the
    parameters and losses of `steps` calls of one step, bit for bit."""
    x, t = (v.astype(np.float32) for v in batch(23, 70))
    a, b = xt.CostModel(0, seed=5), xt.CostModel(0, seed=5)
    h = a.train(x, t, steps, 3e-3)
    hb = np.concatenate([b.train(x, t, 1, 3e-3) for _ in range(steps)])
    assert np.array_equal(h, hb) and np.array_equal(a.get_params(), b.get_params())
    a.close()
    b.close()
