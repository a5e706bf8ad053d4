"""The flux kernel's face lists at the edges of its blocks (runs on an MI355X).

A block takes each face of its 64, 128 or 256 cells once and shares the flux
through LDS, so meshes that end one cell before, at and after a block, quads
(four faces a cell) and the switch from two threads a cell to one (262,144
cells) are compared with the oracle. Rusanov runs the same IEEE operations on
both sides: bit-exact, for the interior and boundary sums apart and together.
"""
import numpy as np
import pytest

from test_gpu_parity import pair

pytestmark = pytest.mark.gpu

BCS = [("left", "upt", {"u": (0.4, 0.1), "p": 1.0, "T": 1.0 / 287.0}), ("right", "p_out", {"p": 0.9}),
       ("top", "wall_adiabatic", {}), ("bottom", "symmetry", {})]


def random_state(n, seed):
    rng = np.random.default_rng(seed)
    rho, u, v, p = (rng.uniform(a, b, n) for a, b in ((0.5, 2.0), (-1.0, 1.0), (-1.0, 1.0), (0.4, 2.0)))
    return np.stack([rho, rho * u, rho * v, p / 0.4 + 0.5 * rho * (u * u + v * v)], 1)


@pytest.mark.parametrize("kind,nx,ny", [("cartesian", 7, 9), ("cartesian", 8, 8), ("cartesian", 5, 13),
                                        ("cartesian", 1, 255), ("cartesian", 257, 1), ("cartesian_tri", 31, 1),
                                        ("cartesian_tri", 8, 8), ("cartesian_tri", 3, 43),
                                        ("cartesian_tri", 512, 256), ("cartesian_tri", 513, 256)])
def test_residual_parts_at_block_edges(mlr, oracle, kind, nx, ny):
    dev, orc, m = pair(mlr, oracle, kind, nx, ny, recon="FO", riemann="Rusanov", bcs=BCS, p_ref=1.0,
                       T_ref=1.0 / 287.0, rho_ref=1.0)
    U = random_state(m.n_cells, nx + ny)
    want = {k: orc.calc_rhs_parts(U, k) for k in (1, 2, 3)}
    for block in (64, 128, 256):
        dev.set_tune(0, block, 256)
        for parts, r in want.items():
            assert np.array_equal(dev.calc_rhs_of(U, parts), r), (block, parts)
