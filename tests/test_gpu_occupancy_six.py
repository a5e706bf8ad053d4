"""Plain TENO at the 6-wave occupancy target, whose members' loads are kept
apart (runs on an MI355X): residual and states of the other targets, bit for
bit, alone and in ensembles, on meshes ending inside and at a 64-cell block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])
SIZES = [(4, 4), (8, 4), (8, 8), (13, 11), (29, 31)]


def numerics(mlr, **kw):
    return mlr.numerics(order=2, teno_variant="corrected", cfl=0.4, **kw)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_solver(mlr, nx, ny):
    out = []
    for occ in (0, 6):
        s = mlr.Solver(gen=mlr.mesh_gen("cartesian_tri", nx, ny, 1.0, 1.0, 0.2, 5), num=numerics(mlr))
        s.init_quadrant(0.5, 0.5, QUADRANT)
        s.set_tune(occ, 128, 128)
        out.append((s.calc_rhs(), s.run_steps(4), *s.state()))
    assert all(np.array_equal(a, b) for a, b in zip(*out))


def test_ensemble(mlr):
    gens = [mlr.mesh_gen("cartesian_tri", nx, ny, 1.0, 1.0, 0.2, 5) for nx, ny in SIZES]
    out = []
    for occ in (0, 6):
        e = mlr.Ensemble(gens, numerics(mlr))
        for k in range(len(gens)):
            e.init_quadrant(k, 0.5, 0.5, QUADRANT)
        e.set_tune(occ, 128)
        e.run_steps(4)
        out.append([e.state(k)[0] for k in range(len(gens))])
    assert all(np.array_equal(a, b) for a, b in zip(*out))
