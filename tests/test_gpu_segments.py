"""Lines solved in segments (solve_impl.hpp) against the oracle, bit for bit.

Sizes around the cuts: lines too short to be cut, just long enough, several
segments with a ragged last one, tiles with a ragged last line, and a line
beyond one tile.  Data on which a segment's warm-up cannot reproduce the
sequential state (constants, zeros after data, an impulse, infinities, NaN)
and numerators whose two-operation division would underflow: there the
kernel has to notice and solve the line in one piece.
"""
import numpy as np
import pytest

from oracle import OracleSpline

pytestmark = pytest.mark.gpu


def _data(kind, shape, rng):
    f = rng.standard_normal(shape)
    if kind == "noise":
        return f
    if kind == "constant":
        return np.broadcast_to(rng.standard_normal(shape[:-1] + (1,)), shape).copy()
    if kind == "constant_first":
        return np.broadcast_to(rng.standard_normal((1,) + shape[1:]), shape).copy()
    if kind == "zero_tail":
        f[..., shape[-1] // 3:] = 0.0
        return f
    if kind == "impulse":
        f[:] = 0.0
        f.flat[0] = 1.0
        f.flat[-1] = -0.0
        return f
    if kind == "tiny":
        return f * 1e-285
    if kind == "huge":
        return f * 1e290
    if kind == "nonfinite":
        f.flat[f.size // 2] = np.nan
        f.flat[f.size // 5] = np.inf
        return f
    raise ValueError(kind)


KINDS = ["noise", "constant", "constant_first", "zero_tail", "impulse", "tiny", "huge", "nonfinite"]

# order, shape, periodic
GRIDS = [
    (3, (95,), "0"), (3, (97,), "0"), (3, (1000,), "0"), (3, (1001,), "1"), (5, (700,), "0"), (6, (515,), "1"),
    (7, (900,), "0"), (7, (640,), "1"), (2, (259,), "1"), (4, (333,), "0"), (1, (200,), "0"),
    (3, (70, 130), "00"), (3, (257, 65), "10"), (5, (129, 200), "01"), (4, (40, 39, 67), "010"),
    (3, (130, 33, 34), "100"), (2, (17, 16, 260), "001"),
    # beyond one tile: chunks of one line, of lines in a row and side by side
    (3, (25000,), "0"), (3, (21000,), "1"), (5, (20481,), "0"), (6, (22528,), "1"), (1, (30000,), "0"),
    (3, (5, 25001), "00"), (3, (5203, 67), "00"), (4, (5121, 66), "10"), (2, (20600, 3), "10"),
]


@pytest.mark.parametrize("order,shape,periodic", GRIDS, ids=lambda v: str(v).replace(" ", ""))
def test_gpu_segments_match_oracle(order, shape, periodic):
    import bsplineinterpolation_amd as amd
    rng = np.random.default_rng(sum(shape) + order)
    per = [c == "1" for c in periodic]
    ranges = [(0.0, 1.0)] * len(shape)
    for kind in KINDS:
        print("segments: order %d %s %s %s" % (order, shape, periodic, kind), flush=True)
        f = _data(kind, shape, rng)
        with np.errstate(all="ignore"):
            want = OracleSpline(order, f, periodic=per, ranges=ranges).control_points()
        got = amd.InterpolationFunction(order, f, periodic=per, ranges=ranges).control_points()
        assert np.array_equal(got, want.reshape(got.shape), equal_nan=True), kind
        # zeros keep their signs (NaN signs are not fixed by IEEE 754)
        ok = ~np.isnan(got)
        assert np.array_equal(np.signbit(got[ok]), np.signbit(want.reshape(got.shape)[ok])), kind


@pytest.mark.parametrize("order,n,periodic", [(3, 45000, False), (6, 24000, True), (5, 60001, False)])
def test_gpu_segments_long_refined(order, n, periodic):
    """Refined lines beyond one tile (FP32, and FP64 arithmetic on FP32
    storage for the periodic order 6) against the FP64 oracle."""
    import bsplineinterpolation_amd as amd
    rng = np.random.default_rng(n)
    t = np.arange(n) / (n if periodic else n - 1)
    f = np.sin(2 * np.pi * 7 * t) + 1e-3 * rng.standard_normal(n)
    x = rng.random((4096, 1))
    want = OracleSpline(order, f, periodic=[periodic], ranges=[(0.0, 1.0)]).eval(x)[0]
    s = amd.InterpolationFunction(order, f, periodic=[periodic], ranges=[(0.0, 1.0)], precision="f32_refined", sweeps=1)
    got = s.eval(x)[0]
    # FP32 control points and weights: a few FP32 roundings of the largest value
    assert np.max(np.abs(got - want)) <= 8 * 2.0 ** -23 * np.max(np.abs(want))


@pytest.mark.parametrize("order,n", [(3, 300), (5, 411)])
def test_gpu_segments_graded_nodes(order, n):
    """Non-uniform lines: no rows of equal factors, every row from memory."""
    import bsplineinterpolation_amd as amd
    rng = np.random.default_rng(n)
    x = np.cumsum(rng.uniform(0.5, 2.0, n))
    f = rng.standard_normal((n, 70))
    y = np.linspace(0.0, 1.0, 70)
    want = OracleSpline(order, f, periodic=[False, False], coords=[x, y]).control_points()
    got = amd.InterpolationFunction(order, f, coords=[x, y]).control_points()
    assert np.array_equal(got, want.reshape(got.shape))
