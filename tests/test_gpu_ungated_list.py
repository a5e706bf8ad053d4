"""Split gated passes: the list of blocks that hold ungated cells (runs on an
MI355X). One block, one list round (4,096 blocks) less and more some, none and
all of the blocks listed: the steps equal those of the one-kernel passes, and
the count of gated cells the recorded decisions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])
EXTRAP = [(z, "extrapolation", {}) for z in ("left", "right", "top", "bottom")]


def network(mlr, level, bias):
    """Smooth where every variable varies by less than 2^level over the stencil; bias shifts the logit."""
    th = np.zeros(mlr.N_PARAMS, np.float32)
    w1, b1 = th[:48 * 64].reshape(48, 64), th[48 * 64:49 * 64]
    for v in range(4):
        w1[v, v], b1[v] = 256.0, -256.0 * (level - 0.5) / 32.0
        th[49 * 64 + v * 64] = 1.0
    th[113 * 64] = -2.0
    th[114 * 64] = -8.0
    th[-1] = bias
    return th


@pytest.mark.parametrize("nx,ny", [(8, 4), (9, 7), (362, 362), (363, 364)])
@pytest.mark.parametrize("bias", [5.0, -1e4, 1e4])
def test_split_equals_one_kernel(mlr, nx, ny, bias):
    gen = mlr.mesh_gen("cartesian_tri", nx, ny, 1.0, 1.0, 0.2, 5)
    num = mlr.numerics(order=2, teno_variant="corrected", cfl=0.4, bcs=EXTRAP)
    got = []
    for split in (True, False):
        s = mlr.Solver(gen=gen, num=num)
        s.init_quadrant(0.5, 0.5, QUADRANT)
        s.set_indicator(network(mlr, -8, bias), 0.9, split=split)
        s.run_steps(3)
        d = s.gate_decisions()
        got.append((s.state()[0], d, s.gated()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
    share = got[0][1].mean()
    assert share == (1.0 if bias > 1e3 else 0.0) if abs(bias) > 1e3 else (nx < 20 or 0.5 < share < 1.0)
