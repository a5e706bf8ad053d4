"""A context's tables in one allocation (runs on an MI355X): sent in one copy up
to 8 MiB (about 32,700 quads or 42,300 triangles), each in its own above.
Residual parts on both sides of the line and on one cell, with fixed states
among the boundaries, bit for bit against the oracle."""
import numpy as np
import pytest

from test_gpu_flux_blocks import BCS, random_state
from test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nx,ny,recon", [("cartesian", 1, 1, "FO"), ("cartesian", 178, 180, "FO"),
                                              ("cartesian", 183, 181, "FO"), ("cartesian_tri", 143, 145, "TENO"),
                                              ("cartesian_tri", 149, 147, "TENO")])
def test_residual(mlr, oracle, kind, nx, ny, recon):
    kw = dict(recon=recon, riemann="Rusanov", bcs=BCS, p_ref=1.0, T_ref=1.0 / 287.0, rho_ref=1.0)
    if recon == "TENO":
        kw.update(order=2, teno_variant="corrected")
    dev, orc, m = pair(mlr, oracle, kind, nx, ny, **kw)
    U = random_state(m.n_cells, nx + ny)
    for parts in (1, 2, 3):
        assert np.array_equal(dev.calc_rhs_of(U, parts), orc.calc_rhs_parts(U, parts)), parts
