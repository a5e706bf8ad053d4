"""The network a training step leaves packed for the next one (runs on an
MI355X). mlp_train returns the parameters after k steps; the next step's rows
are known, so mlp_grad at those parameters, which packs them from scratch,
must give the loss that a longer run records for the step, to the bit, and
the gradient of its update. Group by group: a group left as it was a step
before gives another loss (the backward copy of W2 shows in the update).

The update is repeated in FP32 from that gradient. The two sides take
1 - 0.999^k from powf and numpy, whose last bits may differ: 6e-5 of it at the
first step, half in the update; 1e-4 of the rate and a rounding of the
parameter bound the entries."""
import numpy as np
import pytest

from oracle import indicator_ref as ir
from test_gpu_indicator import _small_dataset
from test_gpu_training_batches import rows

pytestmark = pytest.mark.gpu

GROUPS = dict(W1=(0, ir.OFF_B1), b1=(ir.OFF_B1, ir.OFF_W2), W2=(ir.OFF_W2, ir.OFF_B2), b2=(ir.OFF_B2, ir.OFF_W3),
              w3=(ir.OFF_W3, ir.OFF_B3), b3=(ir.OFF_B3, ir.N_PARAMS))


@pytest.mark.parametrize("batch", [33, 1025])
def test_each_step_continues_the_last(mlr, batch):
    from mallard_amd import indicator as ind
    ds, y = _small_dataset(mlr, n_cases=3, nx=16)
    pool = ind.make_pool(y, seed=2)
    lr, seed, steps = np.float32(2e-3), 7, 4
    kw = dict(pos_w=1.0, neg_w=4.0)
    th = [ind.init_params(3)]
    hist = np.zeros(0, np.float32)
    for k in range(1, steps + 1):
        p, h = mlr.mlp_train(th[0], ds, pool, k, batch, float(lr), seed=seed, **kw)
        assert np.array_equal(h[:k - 1], hist)  # a longer run repeats the shorter one
        th.append(p)
        hist = np.asarray(h, np.float32)
    b1, b2 = np.float32(0.9), np.float32(0.999)
    m, v = np.zeros_like(th[0]), np.zeros_like(th[0])
    for k in range(steps):
        idx = rows(pool, seed, k, batch)
        g, loss = mlr.mlp_grad(th[k], ds, idx, **kw)
        assert hist[k] == np.float32(loss), k
        m = b1 * m + (np.float32(1) - b1) * g
        v = b2 * v + (np.float32(1) - b2) * g * g
        c1, c2 = np.float32(1) - b1 ** np.float32(k + 1), np.float32(1) - b2 ** np.float32(k + 1)
        want = th[k] - lr * (m / c1) / (np.sqrt(v / c2) + np.float32(1e-8))
        for name, (a, e) in GROUPS.items():
            off = np.abs(th[k + 1][a:e] - want[a:e])
            assert (off <= 1e-4 * lr + 2.0 ** -23 * np.abs(want[a:e])).all(), (k, name, off.max() / lr)
            if k:
                stale = th[k].copy()
                stale[a:e] = th[k - 1][a:e]
                assert np.float32(mlr.mlp_grad(stale, ds, idx, **kw)[1]) != hist[k], (k, name)
