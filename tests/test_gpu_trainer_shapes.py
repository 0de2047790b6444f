"""GPU test of the trainer's gradient and prediction at the edges of their
work split: a wave takes 32 samples at a time, a block four waves, a wave takes
several groups from 32 768 samples on, and from 262 113 there are two blocks
per CU.

Tolerance: the targets lie well above the predictions, so no parameter's sum
over the samples loses digits by cancellation beyond its own size; a sample's
FP32 terms carry a few hundred roundings of 2^-24 at most and the tanh and
exp units' 2^-22, about 3e-6 together, and 2e-5 of the largest gradient entry
leaves room for the longest sums."""
import numpy as np
import pytest

import d3q19
import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,count", [(0, 1), (3, 31), (0, 32), (5, 33), (0, 127), (1, 128), (7, 129), (0, 4097),
                                         (11, 65535), (0, 65536), (2, 65537), (9, 131073), (0, 200001),
                                         (1, 262113), (0, 262144), (3, 300007)])
def test_gradient_and_prediction_at_split_edges(first, count):
    rng = np.random.default_rng(count)
    p = d3q19.closure_params(seed=5)
    p[M.B1:M.W2] = rng.uniform(-0.5, 0.5, 32)
    p[M.B2:M.W3] = rng.uniform(-0.5, 0.5, 32)
    p[M.B3] = 0.2
    n = first + count + 3
    X = rng.standard_normal((n, 10)).astype(np.float32)
    y = (3.0 + rng.random(n)).astype(np.float32)
    with d3q19.Trainer(n, p) as tr:
        tr.add_samples(X, y)
        loss, g = tr.grad(first, count)
        again = tr.grad(first, count)
        pred = tr.predict(first, count)
    sl = slice(first, first + count)
    loss_ref, g_ref = M.loss_and_grad(p, X[sl], y[sl])
    assert abs(loss - loss_ref) < 2e-5 * loss_ref
    assert np.max(np.abs(g - g_ref)) < 2e-5 * np.abs(g_ref).max()
    assert loss == again[0] and np.array_equal(g, again[1])
    ref = M.nut(p, X[sl].astype(np.float64))
    assert np.max(np.abs(pred - ref)) < 1e-5 * np.abs(ref).max()
