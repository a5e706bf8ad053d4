"""The positivity scaling of TENO face states where it acts (runs on an
MI355X): a rough state near vacuum, one and two points per face, so that the
quad's lanes hold one or two limits each. Face states bit-exact against the
oracle."""
import numpy as np
import pytest

from test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,nx,ny", [(1, 9, 7), (2, 8, 4), (2, 13, 11), (3, 12, 10)])
def test_face_states_near_vacuum(mlr, oracle, order, nx, ny):
    dev, orc, m = pair(mlr, oracle, "cartesian_tri", nx, ny, recon="TENO", order=order, teno_variant="corrected")
    rng = np.random.default_rng(order)
    n = m.n_cells
    rho, p = np.exp(rng.uniform(np.log(1e-6), np.log(2.0), (2, n)))
    u, v = rng.uniform(-3.0, 3.0, (2, n))
    U = np.stack([rho, rho * u, rho * v, p / 0.4 + 0.5 * rho * (u * u + v * v)], 1)
    fv = dev.calc_face_values(U)
    orc.calc_rhs(U)
    fo = orc.face_values(dev.Q)
    written = ~np.isnan(fv)
    assert np.array_equal(fv[written], fo[written])
    f = fv[written].reshape(-1, 4)
    pf = 0.4 * (f[:, 3] - 0.5 * (f[:, 1] ** 2 + f[:, 2] ** 2) / f[:, 0])
    # some cells were scaled to the floor, and none lies below it
    assert (np.minimum(f[:, 0], pf) < 1e-9).any() and f[:, 0].min() > 0.0
