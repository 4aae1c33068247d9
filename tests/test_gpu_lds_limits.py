"""Lines whose tiles take nearly all LDS of a workgroup, and the first ones
that are cut into chunks instead, against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import OracleSpline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,n,periodic", [
    (1, 20334, False), (1, 20335, False), (1, 20336, False), (3, 20218, False), (3, 20219, False), (3, 20228, False),
    (3, 20229, False), (5, 20021, False), (5, 20022, False), (7, 19732, False), (7, 19733, False), (3, 20287, True),
    (3, 20288, True), (3, 20289, True), (6, 20131, True),
])
def test_gpu_lines_at_the_tile_limit(order, n, periodic):
    import bsplineinterpolation_amd as amd
    f = np.random.default_rng(n).standard_normal(n)
    kw = dict(periodic=[periodic], ranges=[(0.0, 1.0)])
    want = OracleSpline(order, f, **kw).control_points()
    got = amd.InterpolationFunction(order, f, **kw).control_points()
    assert np.array_equal(got, want.reshape(got.shape))


@pytest.mark.parametrize("n", [20334, 20335, 20336])
def test_gpu_graded_lines_at_the_tile_limit(n):
    import bsplineinterpolation_amd as amd
    rng = np.random.default_rng(n)
    x = np.cumsum(rng.uniform(0.5, 2.0, n))
    f = rng.standard_normal(n)
    want = OracleSpline(3, f, periodic=[False], coords=[x]).control_points()
    got = amd.InterpolationFunction(3, f, coords=[x]).control_points()
    assert np.array_equal(got, want.reshape(got.shape))


@pytest.mark.parametrize("shape", [(2, 6755), (2, 6756), (2, 6757), (2, 6758), (2, 6759), (3, 20219), (6755, 2), (10133, 2)])
def test_gpu_few_lines_at_the_tile_limit(shape):
    import bsplineinterpolation_amd as amd
    f = np.random.default_rng(sum(shape)).standard_normal(shape)
    kw = dict(periodic=[False, False], ranges=[(0.0, 1.0)] * 2)
    want = OracleSpline(1, f, **kw).control_points()
    got = amd.InterpolationFunction(1, f, **kw).control_points()
    assert np.array_equal(got, want.reshape(got.shape))


@pytest.mark.parametrize("order,n", [(1, 40686), (1, 40687), (1, 40688), (3, 40613), (3, 40620), (3, 40621)])
def test_gpu_refined_lines_at_the_tile_limit(order, n):
    import bsplineinterpolation_amd as amd
    f = np.random.default_rng(n).standard_normal(n)
    kw = dict(periodic=[False], ranges=[(0.0, 1.0)])
    want = OracleSpline(order, f, **kw).control_points()
    got = amd.InterpolationFunction(order, f, precision="f32_refined", sweeps=2, **kw).control_points()
    # a refined control point is the FP64 one rounded to FP32, up to an error
    # of the last correction far below an FP32 rounding of the largest value
    assert np.max(np.abs(got - want.reshape(got.shape))) <= 2.0 ** -23 * np.max(np.abs(want))


@pytest.mark.parametrize("shape,growth,cells", [((6000, 70), 1.05, 200), ((5500, 64), 1.08, 100), ((5200, 33), 1.05, 200)])
def test_gpu_long_lines_with_long_warm_ups(shape, growth, cells):
    """Lines side by side, too long for a tile, on nodes whose factors fade so
    slowly that 32 lines of a chunk and its warm-up would not fit LDS."""
    import bsplineinterpolation_amd as amd
    rng = np.random.default_rng(shape[0])
    i = np.arange(shape[0])
    steps = growth ** np.minimum(i % (2 * cells), 2 * cells - i % (2 * cells)).astype(float)
    x = np.concatenate([[0.0], np.cumsum(steps[1:])])
    y = np.linspace(0.0, 1.0, shape[1])
    f = rng.standard_normal(shape)
    want = OracleSpline(7, f, periodic=[False, False], coords=[x, y]).control_points()
    got = amd.InterpolationFunction(7, f, coords=[x, y]).control_points()
    assert np.array_equal(got, want.reshape(got.shape))
