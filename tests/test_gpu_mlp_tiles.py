"""The classifier's fused forward and gradient kernels (64 samples per step, at most 512 workgroups)
against the CPU restatement oracle/mlp.py at the edges of their tiles: one sample, one below / at /
above a tile, and more tiles than workgroups.  FP32 against float64: sums of at most 64 products
per unit and two levels over the samples keep every quantity within a few hundred units of 2^-24 of
its largest term (1e-5 of the largest entry allows 168)."""
import numpy as np
import pytest

import mlp as mlp_oracle
import precision as pr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 129, 512 * 64 + 5])
def test_forward_and_gradient_at_tile_edges(n):
    print("mlp tiles n=%d" % n, flush=True)
    rng = np.random.default_rng(n)
    params = (rng.standard_normal(pr.N_PARAMS) * 0.2).astype(np.float32)
    x = rng.standard_normal((n, pr.N_FEATURES)).astype(np.float32)
    y = rng.integers(0, 3, n).astype(np.int32)
    cw = np.array([0.5, 1.0, 2.0], dtype=np.float32)
    model = pr.PrecisionMLP(params, np.zeros(16), np.ones(16))
    p64, x64 = params.astype(np.float64), x.astype(np.float64)
    np.testing.assert_allclose(model.probabilities(x), mlp_oracle.forward(p64, x64)[0], atol=2e-6)
    loss, g = model.loss_grad(x, y, cw)
    lref, gref = mlp_oracle.loss_grad(p64, x64, y, cw.astype(np.float64))
    assert loss == pytest.approx(lref, rel=1e-5)
    assert np.abs(g - gref).max() <= 1e-5 * max(np.abs(gref).max(), 1e-6)
    loss2, g2 = model.loss_grad(x, y, cw)
    assert loss2 == loss and np.array_equal(g, g2)
