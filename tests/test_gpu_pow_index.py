"""The device power where its table index is decided (runs on an MI355X): at,
beside and around the 16 thresholds 2^((j + 1/2)/16), for every binade and
special operand the same bits as on the host, whose index comes from the
thresholds alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 0.5, 2.0, 2.0 ** -1021, 2.0 ** 1000])
def test_same_bits_around_the_thresholds(mlr, scale):
    t = 2.0 ** ((np.arange(-8, 8) + 0.5) / 16)
    d = np.concatenate([[0.0], np.geomspace(1e-16, 1e-2, 57)])
    x = (t[:, None, None] * (1.0 + np.array([-1.0, 1.0])[None, :, None] * d)).ravel() * scale
    for y in (1.0 / 7.0, 0.4 / 2.8, 7.000000000000002, -3.25, 1e-3):
        a, b = mlr.probe_math(2, x, np.full_like(x, y)), mlr.host_pow(x, np.full_like(x, y))
        assert np.array_equal(a.view(np.int64), b.view(np.int64))


def test_special_operands(mlr):
    s = np.array([0.0, -0.0, 1.0, -1.0, np.inf, -np.inf, np.nan, 2.0, -2.0, 3.0, -3.0, 0.5, 5e-324, -1e-310, 1e308,
                  -1e308, 1.0 / 7.0, 1.0 + 2.0 ** -52, 1.0 - 2.0 ** -53])
    x, y = (a.ravel() for a in np.meshgrid(s, s))
    a, b = mlr.probe_math(2, x, y), mlr.host_pow(x, y)
    assert np.array_equal(np.isnan(a), np.isnan(b))
    assert np.array_equal(a[~np.isnan(a)].view(np.int64), b[~np.isnan(b)].view(np.int64))
