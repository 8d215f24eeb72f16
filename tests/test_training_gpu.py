"""Training on the GPU step by step: gradients of large batches (nine taps per
workgroup), the Adam update, the bf16 weights it keeps, and runs longer than one
group of steps.
"""
import os
import sys

import numpy as np
import pytest

from conftest import ROOT, rel

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import cnn_oracle as K  # noqa: E402

pytestmark = pytest.mark.gpu

LAYER = 27 * 32 * 32 + 32
NINE_TAP_ROWS = 170 * 4096  # voxels in all above which a weight gradient takes nine taps per workgroup


def samples(count, V, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((count, V))
    return a * 2.0, 0.6 * a + 0.1 * rng.standard_normal((count, V))


def test_gradient_of_a_large_batch(P, gpu_available):
    """128 samples, two distinct ones in turn: every sample's share is the
    two-sample batch's divided by 64, a power of two, so rounding to bf16 is the
    same and the sums differ in FP32 order alone (a million terms in chains of
    128 and 250: 2^-24 sqrt(378) = 1.2e-6 of the norm, 1e-5 asked).  7980 voxels
    per sample end inside the weight gradient's 256-row blocks.  The two-sample
    batch (three taps) against the oracle as in test_cnn_gpu.py."""
    grid, batch = (20, 21, 19), 128
    V = grid[0] * grid[1] * grid[2]
    assert 2 * V < NINE_TAP_ROWS < batch * V
    print(f"gradient of {batch} samples on {grid}", flush=True)
    a, t = samples(2, V, 3)
    with P.WarmStartNet(grid, max_batch=batch, seed=5) as net:
        params = net.get_params()
        loss2, g2 = net.gradient(a, t)
        loss, g = net.gradient(np.tile(a, (batch // 2, 1)), np.tile(t, (batch // 2, 1)))
    ref = K.network(grid, params, a, t)
    assert abs(loss2 - ref["loss"]) < 1e-4 * ref["loss"] and abs(loss - loss2) < 1e-6 * loss2
    for l in range(4):
        s = slice(l * LAYER, (l + 1) * LAYER)
        assert rel(g2[s], ref["grads"][s]) < 2e-2, (l, rel(g2[s], ref["grads"][s]))
        assert rel(g[s], g2[s]) < 1e-5, (l, rel(g[s], g2[s]))


def test_training_is_gradient_and_adam_step_by_step(P, gpu_available):
    """Each step against gradient() of a second network that is given the
    parameters (and so rounds its weights itself) and Adam in FP32 on the host:
    a few roundings of the update (1e-5 of the learning rate) and of the
    parameter."""
    grid, lr = (9, 10, 11), 2e-3
    a, t = samples(1, 990, 4)
    with P.WarmStartNet(grid, max_batch=1, seed=6) as net, P.WarmStartNet(grid, max_batch=1, seed=7) as other:
        net.set_data(a, t)
        m = v = np.zeros(4 * LAYER + 1, np.float32)
        b1, b2, one = np.float32(0.9), np.float32(0.999), np.float32(1)
        for step in range(1, 5):
            p = net.get_params()
            other.set_params(p)
            want_loss, g = other.gradient(a, t)
            loss = net.train(1, 1, lr=lr, seed=step)
            print(f"step {step}: loss {loss[0]:.6f}", flush=True)
            assert loss[0] == want_loss
            m, v = b1 * m + (one - b1) * g, b2 * v + (one - b2) * g * g
            c1, c2 = one - b1 ** np.float32(step), one - b2 ** np.float32(step)
            want = p - np.float32(lr) * (m / c1) / (np.sqrt(v / c2) + np.float32(1e-8))
            got = net.get_params()
            live = g != 0  # of the 57121 parameters that are not padding
            assert 50000 < live.sum() <= 57121 and np.array_equal(got[~live & (m == 0)], p[~live & (m == 0)])
            assert np.abs(got - want).max() < 1e-5 * lr + 2.0 ** -23 * np.abs(p).max(), np.abs(got - want).max()


def test_weights_kept_by_training_are_the_parameters(P, gpu_available):
    """After training, a network that is given the parameters predicts and
    differentiates bit for bit alike: both bf16 orders of every layer are kept."""
    grid = (13, 8, 9)
    a, t = samples(5, 936, 8)
    with P.WarmStartNet(grid, max_batch=4, seed=6) as net, P.WarmStartNet(grid, max_batch=4, seed=7) as other:
        net.set_data(a, t)
        before = net.predict(a)
        net.train(7, 4, lr=2e-3, seed=1)
        other.set_params(net.get_params())
        got, want = net.predict(a), other.predict(a)
        assert np.array_equal(got, want) and not np.array_equal(got, before)
        (l0, g0), (l1, g1) = net.gradient(a[:4], t[:4]), other.gradient(a[:4], t[:4])
        assert l0 == l1 and np.array_equal(g0, g1)


def test_training_over_several_groups_of_steps(P, gpu_available):
    """Steps are queued in groups that leave 4M partial losses on the device: 4
    steps at max_batch 16384, 1024 at max_batch 1, whose runs are bitwise alike."""
    grid = (3, 2, 4)
    a, t = samples(7, 24, 9)
    runs = []
    for max_batch in (1, 16384):
        with P.WarmStartNet(grid, max_batch=max_batch, seed=6) as net:
            net.set_data(a, t)
            runs.append((net.train(10, 1, lr=2e-3, seed=3), net.get_params()))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
    assert len(set(runs[0][0])) == 10
