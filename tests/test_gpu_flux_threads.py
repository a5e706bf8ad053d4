"""Flux blocks of 256 cells with two threads per cell, up to 131,072 cells, and
with one above (runs on an MI355X). A step's first pass joins the time step
from eight waves' maxima: steps against the same steps one call at a time,
with and without the limiter, bit for bit; and against 64-cell blocks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])


@pytest.mark.parametrize("kind,nx,ny", [("cartesian", 1, 1), ("cartesian", 255, 1), ("cartesian", 257, 1),
                                        ("cartesian", 61, 47), ("cartesian_tri", 256, 256),
                                        ("cartesian_tri", 257, 256)])
@pytest.mark.parametrize("positivity", [False, True])
def test_steps(mlr, kind, nx, ny, positivity):
    num = mlr.numerics(recon="FO", positivity=positivity, cfl=0.4)
    a, b, c = (mlr.Solver(gen=mlr.mesh_gen(kind, nx, ny), num=num) for _ in range(3))
    for s, block in ((a, 256), (b, 256), (c, 64)):
        s.set_tune(0, block, 256)
        s.init_quadrant(0.5, 0.5, QUADRANT)
    dts = a.run_steps(3)
    want = []
    for _ in range(3):
        want.append(b.calc_dt())
        b.take_step()
    assert np.array_equal(dts, np.array(want)) and np.array_equal(dts, c.run_steps(3))
    for s in (b, c):
        assert np.array_equal(a.state()[0], s.state()[0]) and np.array_equal(a.state()[1], s.state()[1])
