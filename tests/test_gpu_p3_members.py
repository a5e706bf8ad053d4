"""TENO at p = 3 outside the streamed pass (runs on an MI355X): other stencil
sizes, gated passes and ensembles run the members' runtime loop. Residuals
against the oracle (Rusanov: the same IEEE operations, bit for bit), gated
steps with a network that never fires against the plain ones, and ensembles
against their cases alone."""
import numpy as np
import pytest

from test_gpu_parity import pair
from test_gpu_flux_blocks import random_state

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])
EXTRAP = [(z, "extrapolation", {}) for z in ("left", "right", "top", "bottom")]


def network(mlr, bias):
    th = np.random.default_rng(4).normal(0.0, 0.2, mlr.N_PARAMS).astype(np.float32)
    th[-1] = bias
    return th


@pytest.mark.parametrize("nx,ny,factor", [(8, 4, 1.5), (9, 7, 2.5), (8, 8, 3.0), (40, 37, 2.5)])
def test_residual_at_other_stencil_sizes(mlr, oracle, nx, ny, factor):
    dev, orc, m = pair(mlr, oracle, "cartesian_tri", nx, ny, 1.0, 1.0, 0.2, 3, recon="TENO", order=3,
                       teno_variant="corrected", riemann="Rusanov", stencil_factor=factor)
    assert dev.M == round(10 * factor)
    U = random_state(m.n_cells, nx + ny)
    assert np.array_equal(dev.calc_rhs_of(U), orc.calc_rhs(U))


@pytest.mark.parametrize("nx,ny", [(8, 4), (11, 9), (40, 37)])
@pytest.mark.parametrize("every_stage", [True, False])
def test_gated_steps(mlr, nx, ny, every_stage):
    gen = mlr.mesh_gen("cartesian_tri", nx, ny, 1.0, 1.0, 0.2, 5)
    num = mlr.numerics(order=3, teno_variant="corrected", cfl=0.4, bcs=EXTRAP)
    plain, never, some = (mlr.Solver(gen=gen, num=num) for _ in range(3))
    never.set_indicator(network(mlr, -1e4), 0.9, every_stage=every_stage)
    some.set_indicator(network(mlr, 2.2), 0.9, every_stage=every_stage)
    ens = mlr.Ensemble([gen, mlr.mesh_gen("cartesian_tri", nx, ny, 1.0, 1.0, 0.2, 6)], num)
    ens.set_indicator(network(mlr, 2.2), 0.9, every_stage=every_stage)
    for s in (plain, never, some):
        s.init_quadrant(0.5, 0.5, QUADRANT)
    for k in range(2):
        ens.init_quadrant(k, 0.5, 0.5, QUADRANT)
    dts = [s.run_steps(4) for s in (plain, never, some)]
    ens.run_steps(4)
    assert never.gated() == 0 and np.array_equal(dts[0], dts[1])
    assert np.array_equal(plain.state()[0], never.state()[0])
    assert np.array_equal(some.state()[0], ens.state(0)[0])
