"""The gradient kernel at the edges of its 64-sample rounds and its 128 rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 8191, 8192, 8193, 20000])
def test_gradient_sizes(bt, oracle, n):
    rng = np.random.default_rng(n)
    p = (0.4 * rng.standard_normal(1377)).astype(np.float32)
    x = rng.random((n, 8)).astype(np.float32)
    y = rng.standard_normal(n).astype(np.float32)
    t = bt.Treecode(0.01, 0.5, 64)
    t.set_mlp_params(p)
    lg, gg = t.mlp_grad(x, y)
    # one step on the whole set moves every parameter by the rate against its gradient
    t.mlp_train(x, y, steps=1, batch=n, lr=1e-3, seed=1)
    moved = t.mlp_params() - p
    t.close()
    lo, go = oracle.mlp_grad(p, x, y)
    assert abs(lg - lo) <= 1e-5 * abs(lo)
    assert np.linalg.norm(gg - go) <= 1e-4 * np.linalg.norm(go)
    big = np.abs(gg) > 1e-5
    assert np.allclose(moved[big], -1e-3 * np.sign(gg[big]), rtol=2e-2)
