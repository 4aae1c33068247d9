"""Proxies whose points are kept in brick order (3D, enough points): equal to
evaluation bit for bit, at the callers' positions, for
FP32 tables, FP32 results and strided results, and the bounds check."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import bsplineinterpolation_amd as amd
    return amd


@pytest.mark.parametrize("shape,order,periodic,npts", [
    ((60, 52, 70), 3, [False, True, False], 1_000_003),
    ((20, 30, 25), 5, [True, False, True], 400_000),   # one radix pass
    ((97, 120, 83), 4, [False, True, False], 262_147),
    ((90, 80, 100), 2, [True, True, True], 900_001),
])
def test_gpu_sorted_proxy_equals_eval(amd, shape, order, periodic, npts):
    import torch
    rng = np.random.default_rng(npts)
    t = amd.InterpolationFunctionTemplate(order, shape, periodic=periodic, ranges=[(0.0, 1.0)] * 3)
    gen = torch.Generator(device="cuda").manual_seed(order)
    q = torch.rand((3, npts), dtype=torch.float64, device="cuda", generator=gen)
    # (the range of a clamped dimension of even order ends before its last node)
    proxy = t.eval_proxy(q.t().contiguous(), bounds=order % 2 == 1)  # points as rows
    for precision in ("f64", "f32_refined"):
        g = t.interpolate(rng.standard_normal(shape), precision=precision)
        want = g.eval(q)[0]
        assert torch.equal(proxy(g), want)
        out = torch.full((npts, 2), 5.0, dtype=torch.float64, device="cuda")
        proxy(g, out=out[:, 0])
        assert torch.equal(out[:, 0], want) and bool((out[:, 1] == 5.0).all())
        out32 = torch.empty(npts, dtype=torch.float32, device="cuda")
        proxy(g, out=out32)
        assert torch.equal(out32, g.eval(q, out_dtype=torch.float32)[0])
    d = [e for e in range(3) if not periodic[e]]
    if d:
        bad = q.clone()
        bad[d[0], npts // 3] = 1.5
        with pytest.raises(amd.DomainError):
            t.eval_proxy(bad.t().contiguous(), bounds=True)
