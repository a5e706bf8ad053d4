"""Tuned launch shapes kept for later solvers (runs on an MI355X): a solver
takes those of an earlier one only where they are its own kernels' shapes. On
one mesh a Legendre solver, tuned where the derived face basis is the faster
one, is followed by a monomial solver, which has no derived basis."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])
EXTRAP = [(z, "extrapolation", {}) for z in ("left", "right", "top", "bottom")]


def solver(mlr, n, basis):
    num = mlr.numerics(basis=basis, order=2, teno_variant="corrected", cfl=0.4, bcs=EXTRAP)
    s = mlr.Solver(gen=mlr.mesh_gen("cartesian_tri", n, n, 1.0, 1.0, 0.2, 5), num=num)
    s.init_quadrant(0.5, 0.5, QUADRANT)
    return s


def test_monomial_after_legendre(mlr):
    for n in (800, 700, 600, 512):  # until the timing picks the derived basis
        s = solver(mlr, n, "legendre")
        picked = s.autotune()[4]
        s.close()
        if picked:
            break
    assert picked
    a, b = solver(mlr, n, "monomial"), solver(mlr, n, "monomial")
    b.set_tune(0, 256, 256)
    dts = a.run_steps(2)
    assert a.tune()[4] == 0
    assert np.array_equal(dts, b.run_steps(2)) and np.array_equal(a.state()[0], b.state()[0])
