"""The library's own choice of grouping against caller order, bit for bit,
where it groups: small tables sorted in one radix pass, gradient cells of
order 4 and 5 (8^3 bricks), bricks whose patch exceeds LDS; every point
layout, result layout and result type.  And a captured call, which keeps to
caller order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import bsplineinterpolation_amd as amd
    return amd


def _points(shape, npts, seed):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand((len(shape), npts), dtype=torch.float64, device="cuda", generator=gen)


def _spline(amd, shape, order, periodic, precision):
    rng = np.random.default_rng(order + sum(shape))
    return amd.InterpolationFunction(order, rng.standard_normal(shape), periodic=periodic,
                                     ranges=[(0.0, 1.0)] * len(shape), precision=precision)


VALUE, D0 = [0, 0, 0], [1, 0, 0]
GRAD = [VALUE, D0, [0, 1, 0], [0, 0, 1]]


@pytest.mark.parametrize("shape,order,periodic,precision,npts,orders", [
    ((24, 31, 20), 5, [False, True, False], "f64", 1_300_003, [VALUE]),            # 24 bricks: one radix pass
    ((48, 48, 48), 5, [False, False, False], "f64", 1_500_000, GRAD),              # 216 bricks
    ((64, 49, 33), 4, [True, False, True], "f32_refined", 700_001, GRAD),          # cells, 280 bricks
    ((100, 90, 80), 5, [False, False, True], "f32_refined", 262_144, GRAD[:2]),    # cells of 35 KB patches
    ((100, 90, 80), 5, [False, False, False], "f64", 262_147, [VALUE, [2, 0, 0]]),  # two launches
    ((230, 210, 190), 7, [False, True, False], "f64", 200_000, [VALUE]),           # no patch in LDS
    ((90, 97, 83), 3, [False, False, False], "f64", 2_000_001, GRAD),
])
def test_gpu_choice_equals_caller_order(amd, shape, order, periodic, precision, npts, orders):
    import torch
    g = _spline(amd, shape, order, periodic, precision)
    q = _points(shape, npts, order)
    want = g.eval(q, orders, group=False)
    assert torch.equal(g.eval(q, orders), want)
    assert torch.equal(g.eval(q, orders, group=True), want)
    # points as rows, results as records
    rec = torch.empty((npts, len(orders)), dtype=torch.float64, device="cuda").t()
    assert torch.equal(g.eval(q.t().contiguous(), orders, out=rec), want)
    f32 = g.eval(q, orders, out_dtype=torch.float32)
    assert torch.equal(f32, g.eval(q, orders, group=False, out_dtype=torch.float32))


def test_gpu_captured_call_keeps_to_caller_order(amd):
    import torch
    g = _spline(amd, (100, 90, 80), 5, [False] * 3, "f64")
    q = _points((100, 90, 80), 400_000, 3)
    want = g.eval(q, GRAD)
    out = torch.empty_like(want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        g.eval(q, GRAD, out=out)
    for i in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        g.eval(q, GRAD[:1])


@pytest.mark.parametrize("precision,order", [("f64", 3), ("f32_refined", 2)])
def test_gpu_record_results_equal_caller_order(amd, precision, order):
    """Large grouped batches store result records and unpack them: rows,
    strided rows, a permuted choice of outputs, FP64 and FP32."""
    import torch
    shape, npts = (70, 61, 83), (1 << 21) + 5
    g = _spline(amd, shape, order, [False, True, False], precision)
    q = _points(shape, npts, 11)
    some = [GRAD[3], GRAD[0], [1, 1, 0], GRAD[2]]
    for orders in (GRAD, some):
        want = g.eval(q, orders, group=False)
        assert torch.equal(g.eval(q, orders, group=True), want)
        wide = torch.full((len(orders), npts + 3), 7.0, dtype=torch.float64, device="cuda")
        assert torch.equal(g.eval(q, orders, group=True, out=wide[:, :npts]), want)
        assert bool((wide[:, npts:] == 7.0).all())
        f32 = g.eval(q, orders, group=True, out_dtype=torch.float32)
        assert torch.equal(f32, g.eval(q, orders, group=False, out_dtype=torch.float32))
