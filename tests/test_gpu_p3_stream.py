"""The p = 3 TENO pass with member tables streamed through LDS (runs on an
MI355X): meshes that end inside, at and after a 64-cell block, 8- and 16-bit
tile positions (8 x 300: a tile of 812 cells, more than 64 KB of LDS with the
ring of members), and stencils left empty near the boundary. Rusanov runs the
same IEEE operations on both sides: bit-exact against the oracle."""
import numpy as np
import pytest

from test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,pos_bytes", [(6, 5, 1), (8, 4, 1), (11, 6, 1), (40, 37, 2), (8, 300, 2)])
def test_residual(mlr, oracle, nx, ny, pos_bytes):
    dev, orc, m = pair(mlr, oracle, "cartesian_tri", nx, ny, 0.2, 3, recon="TENO", order=3, teno_variant="corrected",
                       riemann="Rusanov")
    assert dev.tile_pos_bytes == pos_bytes and dev.K == 10 and dev.M == 20 and dev.Q == 2
    rng = np.random.default_rng(nx)
    n = m.n_cells
    rho, p = rng.uniform(0.5, 2.0, (2, n))
    u, v = rng.uniform(-1.0, 1.0, (2, n))
    U = np.stack([rho, rho * u, rho * v, p / 0.4 + 0.5 * rho * (u * u + v * v)], 1)
    assert np.array_equal(dev.calc_rhs_of(U), orc.calc_rhs(U))
