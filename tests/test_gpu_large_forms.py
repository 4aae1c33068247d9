"""Forms that only large inputs take: the one-pass residual of refined builds
at orders 4 to 7 (from 2^21 control points on) with odd sides, thin and
periodic dimensions, results of grouped batches stored as records (from 2^21
points on) in two dimensions, and grouping in the fixed scratch buffer."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

UNGROUPED, GROUPED = 4, 32


@pytest.fixture(scope="module")
def amd():
    import bsplineinterpolation_amd as amd
    return amd


# The bound is that of half a unit in the last place of FP32 and the FP32
# solve's error on a correction of a few 2^-24 of the largest value: relative
# 1e-4 at these condition numbers.
@pytest.mark.parametrize("shape,order,periodic", [
    ((9, 490, 481), 5, [True, False, False]),
    ((483, 11, 401), 4, [True, True, False]),
    ((129, 131, 127), 5, [False, True, False]),
    ((131, 401, 41), 7, [False, False, True]),
    ((300, 15, 601), 6, [False, True, True]),
    ((13, 403, 403), 7, [True, False, True]),
])
def test_gpu_residual_odd_large(amd, shape, order, periodic):
    assert np.prod(shape) >= 1 << 21
    f = np.random.default_rng(sum(shape) + order).standard_normal(shape)
    kw = dict(periodic=periodic, ranges=[(0.0, 1.0)] * 3)
    want = amd.InterpolationFunction(order, f, **kw).control_points()
    got = amd.InterpolationFunction(order, f, precision="f32_refined", sweeps=3, **kw).control_points()
    bound = 2.0 ** -24 * np.abs(want) + 1e-4 * 2.0 ** -22 * np.abs(want).max()
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) - bound)


def _eval(amd, fn, g, pts, orders, flags, rows):
    import torch
    npts, D = pts.shape
    op = np.ascontiguousarray(np.asarray(orders, np.int32))
    nout = op.shape[0]
    out = torch.full((nout, npts) if rows else (npts, nout), float("nan"), dtype=torch.float64, device="cuda")
    dp = C.POINTER(C.c_double)
    rc = getattr(amd._lib.load(), fn)(g.h, npts, C.cast(pts.data_ptr(), dp), 1, D, nout,
                                      op.ctypes.data_as(C.POINTER(C.c_int32)), C.cast(out.data_ptr(), dp),
                                      npts if rows else 1, 1 if rows else nout, flags,
                                      C.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert rc == 0, amd._lib.load().intp_last_error()
    return out


@pytest.mark.parametrize("rows", [True, False])
@pytest.mark.parametrize("shape,order,periodic,prec", [((700, 901), 3, [True, False], "f64"), ((513, 65), 5, [False, True], "f64"),
                                                       ((300, 301), 2, [False, False], "f32_refined")])
def test_gpu_grouped_records_2d(amd, shape, order, periodic, prec, rows):
    import torch
    f = np.random.default_rng(order).standard_normal(shape)
    g = amd.InterpolationFunction(order, f, periodic=periodic, ranges=[(0.0, 1.0)] * 2, precision=prec)
    gen = torch.Generator(device="cuda").manual_seed(order)
    for npts in ((1 << 21) - 1, 1 << 21, (1 << 21) + 77):
        pts = torch.rand((npts, 2), dtype=torch.float64, device="cuda", generator=gen) * 1.1 - 0.05
        for orders in ([[0, 0], [1, 0], [0, 1]], [[0, 0], [1, 0], [0, 1], [1, 1]], [[0, 0], [1, 1]]):
            got = _eval(amd, "intp_eval", g, pts, orders, GROUPED, rows)
            assert torch.equal(got, _eval(amd, "intp_eval", g, pts, orders, UNGROUPED, rows)), (npts, orders)


@pytest.mark.parametrize("order,shape", [(1, (100, 90, 80)), (3, (200, 200, 200)), (5, (61, 47, 130)), (7, (40, 80, 60))])
def test_gpu_static_grouping(amd, order, shape):
    """Through the fixed buffer: forced at sizes that fit it, by the rule at
    all, below, at and above the least size that uses it by itself."""
    import torch
    f = np.random.default_rng(order).standard_normal(shape)
    g = amd.InterpolationFunction(order, f, periodic=[False, True, False], ranges=[(0.0, 1.0)] * 3)
    gen = torch.Generator(device="cuda").manual_seed(order)
    partials = [[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]]
    for npts in (1, 1000, 40000, (1 << 20) - 1, 1 << 20, (1 << 21) + 5, 5000001):
        pts = torch.rand((npts, 3), dtype=torch.float64, device="cuda", generator=gen)
        for orders in (partials[:1], partials):
            want = _eval(amd, "intp_eval", g, pts, orders, UNGROUPED, False)
            for flags in (0, GROUPED) if npts <= 1 << 20 else (0,):
                assert torch.equal(_eval(amd, "intp_eval_static", g, pts, orders, flags, False), want), (npts, flags)
