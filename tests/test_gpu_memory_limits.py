"""Calls whose extra scratch memory cannot be had: they take the path that
needs none, with the same results.  A child process runs each case with a
limit on what the library may hold (cpp/alloc_limit.cpp)."""
import os
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.alloc_limit.argtypes = [ctypes.c_size_t]
shim.alloc_held.restype = shim.alloc_refused.restype = ctypes.c_size_t
import numpy as np, torch
import bsplineinterpolation_amd as amd
rng = np.random.default_rng(5)
def device(x):
    return torch.from_numpy(x).cuda()
def limit(more):
    # memory beyond what the library holds now (None: no limit)
    torch.cuda.synchronize()
    shim.alloc_limit(2 ** 64 - 1 if more is None else shim.alloc_held() + more)
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("shim") / "liballoclimit.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "cpp", "alloc_limit.cpp"), "-o", so, "-ldl"], check=True)
    return so


def _run(shim, body):
    out = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), shim], cwd=ROOT, capture_output=True,
                         text=True, timeout=110)
    assert out.returncode == 0, out.stdout + out.stderr


@pytest.mark.parametrize("shape,order,periodic,precision", [
    ((60000,), 3, [False], "f64"), ((50000,), 4, [True], "f64"), ((6000, 70), 3, [False, True], "f64"),
    ((70, 30000), 3, [False, False], "f64"), ((90000,), 3, [False], "f32_refined"),
])
def test_gpu_long_lines_without_room_for_chunks(shim, shape, order, periodic, precision):
    """The table and its staging fit, the second table of the chunks does not."""
    _run(shim, """
        shape, order, periodic, precision = %r, %r, %r, %r
        f = device(rng.standard_normal(shape))
        kw = dict(periodic=periodic, ranges=[(0.0, 1.0)] * len(shape), precision=precision, sweeps=1)
        t = amd.InterpolationFunctionTemplate(order, shape, periodic=periodic, ranges=kw["ranges"])
        build = lambda: t.interpolate(f, precision=precision, sweeps=1)
        want = build().control_points()
        # what a build holds at the end is less than a table of chunks more
        n = f.numel()
        need = n * (8 if precision == "f64" else 4 + 8 + 8)
        limit(need + 4096)
        got = build().control_points()
        assert shim.alloc_refused() > 0
        assert np.array_equal(got, want)
    """ % (shape, order, periodic, precision))


@pytest.mark.parametrize("room", ["weights", "weights and order", "all"])
def test_gpu_proxy_without_room_to_sort(shim, room):
    """A proxy's weights fit; what it takes to sort its points does not."""
    _run(shim, """
        room = %r
        n = 1000000
        t = amd.InterpolationFunctionTemplate(4, (60, 50, 40), ranges=[(0.0, 1.0)] * 3)
        spline = t.interpolate(device(rng.standard_normal((60, 50, 40))))
        pts = device(rng.random((n, 3)))
        want = t.eval_proxy(pts)(spline).cpu().numpy()
        weights = (n * 3 * 4 + 255) // 256 * 256 + n * 3 * 5 * 8 + 256
        limit({"weights": weights + 1024, "weights and order": weights + 4 * n + 1024, "all": None}[room])
        got = t.eval_proxy(pts)(spline).cpu().numpy()
        assert (shim.alloc_refused() > 0) == (room != "all")
        assert np.array_equal(got, want)
    """ % room)


def test_gpu_eval_without_room_to_group(shim):
    """Points whose grouping scratch cannot be had stay in caller order."""
    _run(shim, """
        s = amd.InterpolationFunction(5, device(rng.standard_normal((100, 90, 80))), ranges=[(0.0, 1.0)] * 3)
        pts = device(rng.random((1000000, 3)))
        orders = [[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]]
        want = s.eval(pts, orders).cpu().numpy()
        limit(4096)
        got = s.eval(pts, orders).cpu().numpy()
        assert shim.alloc_refused() > 0
        assert np.array_equal(got, want)
    """)
