"""The training step at the edges of its blocks and of its block sum (runs on
an MI355X): one row, a block of 32 rows less and more one, and 32 and 33
blocks (the block sum takes 32 at a time).

Each step's gradient and loss come from mlp_grad on the rows the documented
hash draws; the Adam update is repeated in FP32. The two sides take
c2 = 1 - 0.999^k from powf and numpy, whose last bits may differ: 6e-8 of a
value near 1 is 6e-5 of c2 at the first step, half of that in the update, so
entries agree within 1e-4 of the rate per step."""
import numpy as np
import pytest

from oracle import indicator_ref as ir
from test_gpu_indicator import _small_dataset

pytestmark = pytest.mark.gpu


def rows(pool, seed, step, batch):
    mask = (1 << 64) - 1
    out = []
    for i in range(batch):
        x = (seed * 0x9E3779B97F4A7C15 + step * 0xBF58476D1CE4E5B9 + i * 0x94D049BB133111EB) & mask
        x ^= x >> 30
        x = x * 0xBF58476D1CE4E5B9 & mask
        x ^= x >> 27
        x = x * 0x94D049BB133111EB & mask
        x ^= x >> 31
        out.append(pool[x % len(pool)])
    return np.array(out, np.uint32)


@pytest.mark.parametrize("batch", [1, 31, 32, 33, 1024, 1025])
def test_steps_are_gradient_and_adam(mlr, batch):
    from mallard_amd import indicator as ind
    ds, y = _small_dataset(mlr, n_cases=3, nx=16)
    X, yy = ds.get()
    pool = ind.make_pool(y, seed=2)
    lr, seed, steps = np.float32(2e-3), 7, 3
    th0 = ind.init_params(3)
    got, hist = mlr.mlp_train(th0, ds, pool, steps, batch, float(lr), seed=seed, pos_w=1.0, neg_w=4.0)
    th = th0.copy()
    m, v = np.zeros_like(th), np.zeros_like(th)
    b1, b2 = np.float32(0.9), np.float32(0.999)
    for k in range(steps):
        idx = rows(pool, seed, k, batch)
        g, loss = mlr.mlp_grad(th, ds, idx, pos_w=1.0, neg_w=4.0)
        lr_, gr = ir.loss_grad(th, X[idx], yy[idx], pos_w=1.0, neg_w=4.0)
        assert np.abs(g - gr).max() <= 2e-3 * np.abs(gr).max() and abs(loss - lr_) <= 1e-4 * max(1.0, abs(lr_))
        if k == 0:
            assert hist[0] == np.float32(loss)
        m = b1 * m + (np.float32(1) - b1) * g
        v = b2 * v + (np.float32(1) - b2) * g * g
        c1, c2 = np.float32(1) - b1 ** np.float32(k + 1), np.float32(1) - b2 ** np.float32(k + 1)
        th = th - lr * (m / c1) / (np.sqrt(v / c2) + np.float32(1e-8))
        if k == 0:  # one step: the gradient is the same on both sides
            one, _ = mlr.mlp_train(th0, ds, pool, 1, batch, float(lr), seed=seed, pos_w=1.0, neg_w=4.0)
            assert np.abs(one - th).max() <= 1e-4 * lr
    # the later gradients see parameters apart by rounding: a step moves an entry by at most about the rate
    assert np.median(np.abs(got - th)) <= 1e-3 * lr and np.abs(got - th).max() <= 2 * steps * lr
