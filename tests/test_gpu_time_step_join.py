"""The time step joined by a step's first flux pass (runs on an MI355X): up to
1,024 block maxima of the radii the flux blocks join them, above one block
does. Meshes on both sides of the switch (spectral blocks of 64 and 256
cells), with fixed steps, the limiter and each integrator, against the same
steps taken one call at a time (calc_dt, then take_step), bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])


@pytest.mark.parametrize("nx,ny,spec", [(1, 1, 64), (13, 7, 64), (256, 256, 64), (257, 256, 64), (300, 250, 256)])
@pytest.mark.parametrize("integrator,positivity,dt", [("SSPRK3", False, 0.0), ("RK4", False, 0.0), ("FE", True, 0.0),
                                                      ("SSPRK3", True, 0.0), ("SSPRK3", False, 1e-5)])
def test_steps_equal_single_calls(mlr, nx, ny, spec, integrator, positivity, dt):
    # cfl 0 selects the fixed time step
    num = mlr.numerics(recon="FO", integrator=integrator, positivity=positivity, cfl=0.0 if dt else 0.4, dt=dt)
    a, b = (mlr.Solver(gen=mlr.mesh_gen("cartesian", nx, ny), num=num) for _ in range(2))
    for s in (a, b):
        s.set_tune(0, 128, spec)
        s.init_quadrant(0.5, 0.5, QUADRANT)
    dts = a.run_steps(3)
    want = []
    for _ in range(3):
        want.append(b.calc_dt())
        b.take_step()
    assert np.array_equal(dts, np.array(want))
    assert np.array_equal(a.state()[0], b.state()[0]) and np.array_equal(a.state()[1], b.state()[1])
    assert a.time()[1] == 3 and np.isfinite(a.state()[0]).all()
