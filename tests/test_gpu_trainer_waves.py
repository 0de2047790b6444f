"""GPU test of the trainer where its blocks change from four waves to eight
(32 768 samples, a group of 32 for each of 1 024 waves) and where waves take
second groups (above 65 536), against the oracle in 64 bits, and of predictions
in and around the slices of their copies (64 KiB, 1 MiB, remainders, a first
sample off a multiple of 4).

Tolerance: as for the other sizes (test_gpu_trainer_shapes.py): FP32 terms of
a few hundred roundings of 2^-24 at most, 2e-5 of the largest entry."""
import numpy as np
import pytest

import d3q19
import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,count", [(1, 32767), (0, 32768), (3, 32769), (0, 32993), (2, 65505), (5, 65569),
                                         (7, 98305)])
def test_gradient_where_blocks_grow(first, count):
    rng = np.random.default_rng(count)
    p = d3q19.closure_params(seed=6)
    p[M.B1:M.W2], p[M.B2:M.W3] = rng.uniform(-0.5, 0.5, 32), rng.uniform(-0.5, 0.5, 32)
    X = rng.standard_normal((first + count + 2, 10)).astype(np.float32)
    y = (3.0 + rng.random(len(X))).astype(np.float32)
    with d3q19.Trainer(len(X), p) as tr:
        tr.add_samples(X, y)
        loss, g = tr.grad(first, count)
        before = tr.params()
        assert tr.train(first, count, iterations=1, batch=count, lr=1e-3) == loss
        after = tr.params()
    sl = slice(first, first + count)
    loss_ref, g_ref = M.loss_and_grad(p, X[sl], y[sl])
    assert abs(loss - loss_ref) < 2e-5 * loss_ref
    assert np.max(np.abs(g - g_ref)) < 2e-5 * np.abs(g_ref).max()
    # Adam's first step is lr g / (|g| + eps sqrt(1 - beta2)): lr in size where g is not tiny
    big = np.abs(g_ref) > 1e-3 * np.abs(g_ref).max()
    step = (after - before)[:len(g_ref)][big]
    assert np.max(np.abs(step + 1e-3 * np.sign(g_ref[big]))) < 1e-5


@pytest.mark.parametrize("first,count", [(0, 1), (1, 16383), (0, 16384), (3, 16385), (2, 262144), (1, 262145), (5, 600001)])
def test_predictions_in_slices(first, count):
    rng = np.random.default_rng(count)
    p = d3q19.closure_params(seed=7)
    X = rng.standard_normal((first + count + 1, 10)).astype(np.float32)
    with d3q19.Trainer(len(X), p) as tr:
        tr.add_samples(X, np.zeros(len(X), dtype=np.float32))
        pred = tr.predict(first, count)
    ref = M.nut(p, X[first:first + count].astype(np.float64))
    assert np.max(np.abs(pred - ref)) < 1e-5 * np.abs(ref).max()
