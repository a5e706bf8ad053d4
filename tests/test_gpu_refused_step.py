"""A step whose launch is refused (runs on an MI355X): no TENO kernel takes as
many face points as a face quadrature of order 3 has. The same thread's other
contexts go on working, and the context gives its state and the same error."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUADRANT = np.array([[1.5, 0.0, 0.0, 1.5], [0.5323, 1.206, 0.0, 0.3],
                     [0.138, 1.206, 1.206, 0.029], [0.5323, 0.0, 1.206, 0.3]])


def test_refused_launch_ends_the_capture(mlr):
    gen = mlr.mesh_gen("cartesian_tri", 12, 10, 1.0, 1.0, 0.2, 5)
    s = mlr.Solver(gen=gen, num=mlr.numerics(order=2, teno_variant="corrected", quad_order_face=3))
    s.init_quadrant(0.5, 0.5, QUADRANT)
    s.set_tune(0, 256, 256)
    U = s.state()[0]
    for _ in range(2):
        with pytest.raises(mlr.MallardError, match="invalid argument"):
            s.run_steps(1)
    assert np.array_equal(s.state()[0], U)
    t = mlr.Solver(gen=gen, num=mlr.numerics(order=2, teno_variant="corrected"))
    t.init_quadrant(0.5, 0.5, QUADRANT)
    assert t.run_steps(2).min() > 0.0
