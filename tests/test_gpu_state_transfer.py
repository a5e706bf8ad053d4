"""States to and from the solver's numbering (runs on an MI355X): the GPU
renumbers them, so meshes around one 256-thread block are set, read and
initialised, bit for bit (the primitives against the same operations in numpy).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GAMMA = 1.4
R_GAS = 101325.0 / (298.15 * 1.225)


def primitives(U):
    cv = (R_GAS * GAMMA / (GAMMA - 1.0)) / GAMMA
    rho = U[:, 0]
    u, v = U[:, 1] / rho, U[:, 2] / rho
    e = U[:, 3] / rho - 0.5 * (u * u + v * v)
    p = (GAMMA - 1.0) * rho * e
    return np.stack([u, v, p, e / cv, e + p / rho], 1)


@pytest.mark.parametrize("nx,ny", [(1, 1), (255, 1), (16, 16), (1, 257), (61, 47)])
def test_set_and_read(mlr, nx, ny):
    s = mlr.Solver(gen=mlr.mesh_gen("cartesian", nx, ny), num=mlr.numerics(recon="FO"))
    rng = np.random.default_rng(nx + 7 * ny)
    U = np.concatenate([rng.uniform(0.5, 2.0, (nx * ny, 1)), rng.uniform(-1.0, 1.0, (nx * ny, 2)),
                        rng.uniform(4.0, 6.0, (nx * ny, 1))], 1)
    s.set_state(U)
    got = s.state()
    assert np.array_equal(got[0], U) and np.array_equal(got[1], primitives(U))
    W = rng.uniform(-3.0, 3.0, (nx * ny, 5))
    s.set_state(U, W)
    got = s.state()
    assert np.array_equal(got[0], U) and np.array_equal(got[1], W)


@pytest.mark.parametrize("nx,ny", [(1, 1), (255, 1), (16, 16), (1, 257), (61, 47)])
def test_initial_regions(mlr, nx, ny):
    s = mlr.Solver(gen=mlr.mesh_gen("cartesian", nx, ny), num=mlr.numerics(recon="FO"))
    q = np.array([[1.5, 0.1, 0.2, 1.5], [0.53, 1.2, 0.0, 0.3], [0.14, 1.2, 1.2, 0.03], [0.52, 0.0, 1.2, 0.31]])
    s.init_quadrant(0.47, 0.61, q)
    x, y = np.meshgrid((np.arange(nx) + 0.5) / nx, (np.arange(ny) + 0.5) / ny, indexing="ij")
    w = q[np.where(x >= 0.47, np.where(y >= 0.61, 0, 3), np.where(y >= 0.61, 1, 2))].reshape(-1, 4)
    U, W = s.state()
    assert np.array_equal(U[:, 0], w[:, 0]) and np.array_equal(U[:, 1], w[:, 0] * w[:, 1])
    assert np.array_equal(W[:, :3], w[:, 1:])
    s.init_constant([0.3, -0.2], 0.9, 250.0)
    U, W = s.state()
    assert (U == U[0]).all() and (W == W[0]).all() and W[0, 2] == 0.9 and W[0, 3] == 250.0
