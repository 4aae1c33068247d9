"""The one-pass residual of refined builds (residual_kernel) at the edges of
its tiles and chunks, every order, clamped and periodic.

After three sweeps a control point is the FP64 one rounded to FP32, up to
the last correction's own error: the correction is a few 2^-24 of the
largest value and is solved in FP32, so its error is below 2^-24 times the
solve's relative error, itself below 1e-4 here (orders up to 7: condition
numbers per dimension up to about 10^3, FP32 rounding 6e-8).  The bound is
half a unit in the last place, 2^-24 of the value, plus 1e-4 times 2^-22 of
the largest.  A residual that is wrong anywhere leaves errors of the FP32
solve, 1e-6 and more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import bsplineinterpolation_amd as amd
    return amd


@pytest.mark.parametrize("shape,order,periodic", [
    ((33, 65), 3, [False, False]),
    ((64, 32), 2, [True, False]),
    ((31, 129), 5, [False, True]),
    ((20, 200), 4, [True, True]),
    ((9, 33, 65), 3, [False, False, False]),
    ((70, 32, 64), 5, [False, False, False]),
    ((17, 31, 63), 4, [True, False, True]),
    ((40, 34, 66), 5, [False, True, False]),
    ((16, 64, 20), 2, [False, False, True]),
    ((25, 12, 130), 1, [False, False, False]),
    ((19, 37, 70), 6, [True, True, True]),
    ((24, 36, 16), 7, [False, False, True]),
    ((300, 33, 9), 3, [True, False, False]),
])
def test_gpu_residual_tiles(amd, shape, order, periodic):
    rng = np.random.default_rng(sum(shape) + order)
    f = rng.standard_normal(shape)
    kw = dict(periodic=periodic, ranges=[(0.0, 1.0)] * len(shape))
    want = amd.InterpolationFunction(order, f, **kw).control_points()
    got = amd.InterpolationFunction(order, f, precision="f32_refined", sweeps=3, **kw).control_points()
    bound = 2.0 ** -24 * np.abs(want) + 1e-4 * 2.0 ** -22 * np.abs(want).max()
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) - bound)


@pytest.mark.parametrize("shape,order", [((128, 128, 128), 4), ((64, 200, 165), 6), ((130, 130, 130), 7)])
def test_gpu_residual_large_orders(amd, shape, order):
    """Orders 4 and up take the one pass from 2^21 control points on."""
    rng = np.random.default_rng(order)
    f = rng.standard_normal(shape)
    kw = dict(periodic=[order == 6, False, True], ranges=[(0.0, 1.0)] * 3)
    want = amd.InterpolationFunction(order, f, **kw).control_points()
    got = amd.InterpolationFunction(order, f, precision="f32_refined", sweeps=3, **kw).control_points()
    bound = 2.0 ** -24 * np.abs(want) + 1e-4 * 2.0 ** -22 * np.abs(want).max()
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) - bound)
