"""The launch shape that a context reports before it is tuned (runs on an
MI355X): the neutral choice at every size, and pinned with one entry changed
it is accepted. Meshes on both sides of 262,144 cells, where untuned launches
begin to derive the face basis."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])


@pytest.mark.parametrize("nx,ny", [(20, 20), (362, 362), (363, 363)])
def test_neutral_choice(mlr, nx, ny):
    s = mlr.Solver(gen=mlr.mesh_gen("cartesian_tri", nx, ny, 1.0, 1.0, 0.2, 5),
                   num=mlr.numerics(order=2, teno_variant="corrected"))
    assert s.tune() == (0, 256, 256, 0, 0)
    s.init_quadrant(0.5, 0.5, QUADRANT)
    r = s.calc_rhs()
    assert s.tune() == (0, 256, 256, 0, 0)
    for entry, value in ((0, 6), (0, 5), (1, 64), (2, 128), (3, 6)):
        t = [0, 256, 256, 0, 0]
        t[entry] = value
        s.set_tune(*t)
        assert s.tune() == tuple(t) and np.array_equal(s.calc_rhs(), r)
