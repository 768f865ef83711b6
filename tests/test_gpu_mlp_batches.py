"""The network's row-blocked kernels at the edges of their blocks: one row, a
block less and more one, a slice of the dW2 product with no rows, a batch beyond
one final run of blocks.  Against the float64 restatement with the device's BF16
roundings: an operand on the edge of a BF16 rounding moves its term by 2^-9, so a
block's relative error stays below 2e-3."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 31, 32, 33, 255, 513, 1040])
def test_gradients_and_scores(lib, B):
    from oracle import mlp_ref as R
    net = lib.MLP(seed=3)
    rng = np.random.default_rng(B)
    X = np.abs(rng.standard_normal((B, 8))).astype(np.float32) * 2
    y = (rng.random(B) < 0.4).astype(np.float32)
    net.grad(np.ones((2000, 8), np.float32), np.ones(2000, np.float32))  # stale partial sums
    g, loss = net.grad(X, y, pos_w=2.0)
    p = net.params()
    loss_ref, g_ref, logit = R.forward_backward(p, X, y, pos_w=2.0, bf16=True)
    assert abs(loss - loss_ref) <= 1e-4 * abs(loss_ref)
    for a, b in ((R.OW1, R.OB1), (R.OB1, R.OW2), (R.OW2, R.OB2), (R.OB2, R.OW3), (R.OW3, R.OB3),
                 (R.OB3, R.NP)):
        assert np.linalg.norm(g[a:b] - g_ref[a:b]) <= 2e-3 * np.linalg.norm(g_ref[a:b])
    assert np.abs(net.scores(X) - logit).max() <= 2e-3 * max(1.0, np.abs(logit).max())
    np.testing.assert_array_equal(net.grad(X, y, pos_w=2.0)[0], g)
    net.close()
