"""How a batch's lines are solved (batch.hip): tiles in one launch or by size,
lines cut into segments or whole, strided axes one line per lane.  Control
points are those of single splines bit for bit on any data, and a few splines
together cost about what the largest of them costs alone."""
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _specs(seed, count, dim, lo, hi, orders=(1, 5)):
    rng = random.Random(seed)
    return [dict(order=rng.randint(*orders), shape=tuple(rng.randint(lo, hi) for _ in range(dim)),
                 periodic=[rng.random() < 0.3 for _ in range(dim)], ranges=[(0.0, 1.0)] * dim) for _ in range(count)]


def _batches():
    return {
        "few_short": _specs(1, 12, 2, 16, 120),
        "few_long": _specs(2, 10, 2, 280, 700),
        "few_mixed": _specs(3, 40, 2, 16, 256, (1, 7)) + _specs(4, 6, 3, 8, 64),
        "many_mixed": _specs(5, 1500, 2, 16, 256),       # above 16 tiles per CU: a launch per size
        "many_long": _specs(6, 420, 2, 200, 420),        # strided lines fill the chip
        "three": _specs(7, 40, 3, 12, 150),
        "one_long_axis": _specs(16, 300, 2, 16, 160) + [dict(order=k, shape=shape, periodic=[False] * 2, ranges=[(0.0, 1.0)] * 2)
                                                        for k, shape in ((3, (9, 15000)), (4, (12000, 5)), (5, (14000, 40)))],
        "thin": _specs(8, 30, 2, 700, 1200, (2, 4)) + _specs(9, 30, 3, 8, 24, (6, 7)),
        "many_unequal_lines": _specs(11, 6000, 1, 16, 500) + [dict(order=3, shape=(n,), periodic=[False], ranges=[(0.0, 1.0)])
                                                              for n in (3000, 5000, 9000, 17000)],
        "unequal_lines": _specs(10, 300, 1, 16, 400) + [dict(order=k, shape=(n,), periodic=[p], ranges=[(0.0, 1.0)])
                                                        for k, n, p in ((3, 9000, False), (5, 17000, False), (4, 6000, True),
                                                                        (2, 30000, False))],
    }


def _data(kind, specs, total):
    rng = np.random.default_rng(total)
    if kind == "constant":
        return np.full(total, 0.7372)
    v = rng.standard_normal(total)
    if kind == "zero_tail":
        v[np.arange(total) % 400 >= 60] = 0.0
    return v


@pytest.mark.parametrize("name", ["few_short", "few_long", "few_mixed", "many_mixed", "many_long", "three", "thin", "one_long_axis",
                                  "unequal_lines", "many_unequal_lines"])
def test_gpu_batch_forms_equal_single_splines(name):
    import torch
    import bsplineinterpolation_amd as amd
    specs = _batches()[name]
    batch = amd.Batch(specs)
    sizes = [int(np.prod(s["shape"])) for s in specs]
    first = np.concatenate([[0], np.cumsum(sizes)])
    sample = sorted({int(i) for i in np.linspace(0, len(specs) - 1, 24)} | {int(np.argmax(sizes)), int(np.argmin(sizes))})
    for kind in ("noise", "constant", "zero_tail"):
        v = _data(kind, specs, batch.total)
        batch.build(torch.from_numpy(v).cuda())
        torch.cuda.synchronize()
        for s in sample:
            spec = specs[s]
            one = amd.InterpolationFunction(spec["order"], v[first[s]:first[s + 1]].reshape(spec["shape"]),
                                            periodic=spec["periodic"], ranges=spec["ranges"])
            assert np.array_equal(batch.control_points(s), one.control_points().ravel()), (kind, s, spec)


def _microseconds(build):
    import torch
    best = float("inf")
    for _ in range(20):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        build()
        end.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(end) * 1e3)
    return best


def test_gpu_batch_of_a_few_costs_its_largest():
    """Forty splines are fewer tiles than the chip holds at once: beside the
    longest line there is the start of the workgroups and the contention for
    the caches, less than the line again."""
    import torch
    import bsplineinterpolation_amd as amd
    specs = [dict(order=o, shape=(n, n + 4), periodic=[False] * 2, ranges=[(0.0, 1.0)] * 2)
             for o in (2, 3, 4, 5) for n in range(30, 250, 22)]
    many, one = amd.Batch(specs), amd.Batch([specs[-1]])
    v = torch.randn(many.total, dtype=torch.float64, device="cuda")
    w = v[:one.total].clone()
    us, base = _microseconds(lambda: many.build(v)), _microseconds(lambda: one.build(w))
    print("%d splines %.0f us, the largest %.0f us" % (len(specs), us, base), flush=True)
    assert us <= 2.0 * base


def test_gpu_batch_long_line_beside_short_ones():
    """A launch that gives every line the LDS of the longest holds few at a
    time; side by side they take no longer than one after the other."""
    import torch
    import bsplineinterpolation_amd as amd
    long = dict(order=3, shape=(18000,), periodic=[False], ranges=[(0.0, 1.0)])
    short = _specs(12, 8000, 1, 50, 500)
    us = []
    for specs in ([long], short, short + [long]):
        batch = amd.Batch(specs)
        v = torch.randn(batch.total, dtype=torch.float64, device="cuda")
        us.append(_microseconds(lambda: batch.build(v)))
    print("long %.0f us, short %.0f us, together %.0f us" % tuple(us), flush=True)
    assert us[2] <= us[0] + us[1]


def test_gpu_batch_forms_in_a_graph():
    """The launches side by side, captured and replayed with other values,
    with split lines and without."""
    import torch
    import bsplineinterpolation_amd as amd
    specs = _specs(13, 6000, 1, 50, 400) + [dict(order=3, shape=(n,), periodic=[False], ranges=[(0.0, 1.0)])
                                            for n in (9000, 3000)] + _specs(14, 200, 2, 16, 300) + _specs(15, 10, 3, 8, 90)
    batch, rng = amd.Batch(specs), np.random.default_rng(3)
    q = 8
    po = np.arange(len(specs) + 1) * q
    pts = torch.from_numpy(rng.random((q * len(specs), 3)) * 0.999).cuda()
    vals = torch.from_numpy(rng.standard_normal(batch.total)).cuda()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for split in (False, True):
            plain = batch.run(vals, pts, po, split_lines=split).clone()
            out = torch.empty_like(plain)
            for scale in (1.0, 2.0, 0.5):  # exact scalings
                torch.mul(vals, scale, out=vals)
                torch.mul(plain, scale, out=plain)
                batch.run(vals, pts, po, out=out, graph=True, split_lines=split)
                stream.synchronize()
                assert torch.equal(out, plain), (split, scale)


def test_gpu_batch_long_axis_beside_short_ones():
    """As above, for the tiles of a pass."""
    import torch
    import bsplineinterpolation_amd as amd
    long = dict(order=3, shape=(4, 15000), periodic=[False] * 2, ranges=[(0.0, 1.0)] * 2)
    short = _specs(17, 1500, 2, 128, 160)
    us = []
    for specs in ([long], short, short + [long]):
        batch = amd.Batch(specs)
        v = torch.randn(batch.total, dtype=torch.float64, device="cuda")
        us.append(_microseconds(lambda: batch.build(v)))
    print("long %.0f us, short %.0f us, together %.0f us" % tuple(us), flush=True)
    assert us[2] <= us[0] + us[1]
