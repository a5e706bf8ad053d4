"""The spectral block that tuning picks (runs on an MI355X): where some block
size leaves at most 1,024 maxima, so that a step's first flux pass can join
them, the pick is one that does. Quads on both sides of each size's line."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])


@pytest.mark.parametrize("nx,ny", [(50, 40), (256, 256), (257, 256), (300, 300), (512, 256), (513, 256), (512, 512),
                                   (513, 512)])
@pytest.mark.parametrize("riemann", ["Rusanov", "HLLC"])
def test_maxima_of_the_tuned_block(mlr, nx, ny, riemann):
    s = mlr.Solver(gen=mlr.mesh_gen("cartesian", nx, ny), num=mlr.numerics(recon="FO", riemann=riemann, cfl=0.4))
    s.init_quadrant(0.5, 0.5, QUADRANT)
    block = s.autotune()[2]
    assert block in (64, 128, 256)
    if -(-nx * ny // 256) <= 1024:
        assert -(-nx * ny // block) <= 1024
    assert (s.run_steps(3) > 0.0).all()
