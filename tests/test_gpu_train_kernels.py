"""The training kernels at the batch sizes where their tiling can go wrong: one row, either side of a
wave's 16 rows, of the workspace's 128-row padding, of a gradient slice, and of the rule between four-
and eight-wave workgroups (16,384 rows); and a batch after a larger one in the same workspace.

Tolerances: the oracle rounds to bf16 where the kernels do, so the two differ by f32 summation order
and by the rare activation whose rounding that order flips (one bf16 ulp, 2^-8 relative, of one
element): 1e-2 of a gradient tensor's norm and 2e-3 of the largest output, the bars of the
1,000-row gradient test."""
import numpy as np
import pytest

import feriphys_amd as fa
import mlp_oracle as mo
from gpu_common import announce

pytestmark = pytest.mark.gpu

TENSORS = (("W1", mo.OFF_W1, mo.OFF_B1), ("b1", mo.OFF_B1, mo.OFF_W2), ("W2", mo.OFF_W2, mo.OFF_B2),
           ("b2", mo.OFF_B2, mo.OFF_W3), ("W3", mo.OFF_W3, mo.OFF_B3), ("b3", mo.OFF_B3, mo.OFF_W4),
           ("W4", mo.OFF_W4, mo.OFF_B4), ("b4", mo.OFF_B4, mo.N_PARAMS))


def batch(rows, seed):
    rng = np.random.default_rng(seed)
    return (rng.normal(scale=0.6, size=(rows, 72)).astype(np.float32),
            rng.normal(scale=0.5, size=(rows, 3)).astype(np.float32))


@pytest.mark.parametrize("rows", [1, 15, 17, 127, 129, 513, 16384, 16385])
def test_gradient_at_tile_edges(rows):
    announce(f"training gradient, {rows} rows")
    net = fa.Surrogate(seed=5)
    X, T = batch(rows, rows)
    loss, g, Y = net.grad(X, T)
    lo, go, Yo = mo.loss_and_grad(net.get_params().astype(np.float64), X, T, emulate=True)
    assert abs(loss - lo) <= 1e-3 * lo
    assert np.abs(Y - Yo).max() <= 2e-3 * np.abs(Yo).max()
    for name, a, b in TENSORS:
        assert np.linalg.norm(g[a:b] - go[a:b]) <= 1e-2 * np.linalg.norm(go[a:b]), name


def test_a_smaller_batch_after_a_larger_one():
    """900 and 1,003 rows share a row length of 1,024: nothing of the first may reach the second."""
    announce("training gradient, 1003 then 900 rows")
    X, T = batch(1003, 1)
    net, fresh = fa.Surrogate(seed=5), fa.Surrogate(seed=5)
    net.grad(X, T)
    a, b = net.grad(X[:900], T[:900]), fresh.grad(X[:900], T[:900])
    assert a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


def test_one_adam_step_is_the_gradient_step():
    """From zero moments, Adam's first update is lr g / (|g| + eps sqrt(1 - b2)) with c1 = 1 - b1: the
    batch of a one-sample training set is that sample, whatever rows the hash draws."""
    announce("one Adam step")
    X, T = batch(1, 9)
    net = fa.Surrogate(seed=5)
    p = net.get_params()
    loss, g, _ = net.grad(np.repeat(X, 200, 0), np.repeat(T, 200, 0))
    net.add_samples(X, T)
    losses = net.train(1, batch=200, lr=1e-3, seed=4)
    assert abs(losses[0] - loss) <= 1e-6 * loss
    big = np.abs(g) > 1e-5 * np.abs(g).max()
    assert np.abs((net.get_params() - p)[big] + 1e-3 * np.sign(g[big])).max() <= 2e-6
