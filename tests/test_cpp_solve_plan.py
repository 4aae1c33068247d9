"""The host-side choices of the line solves (solve_plan.hpp), on the CPU, with
the static LDS that the built kernels have."""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bsplineinterpolation_amd", "csrc")
LIB = os.path.join(ROOT, "bsplineinterpolation_amd", "libintp_amd.so")
LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def plan_test(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "solve_plan_test")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + CSRC, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpp", "solve_plan_test.cpp"), os.path.join(CSRC, "setup.cpp"),
                    "-o", exe], check=True)
    return exe


def _static_lds(tmp, kernels):
    """The largest static LDS of the named kernels in the built library."""
    objdump, readelf = os.path.join(LLVM, "llvm-objdump"), os.path.join(LLVM, "llvm-readelf")
    if not (os.path.exists(LIB) and os.path.exists(objdump) and os.path.exists(readelf)):
        pytest.skip("library or LLVM tools not available")
    so = os.path.join(tmp, "lib.so")
    shutil.copy(LIB, so)
    subprocess.run([objdump, "--offloading", so], cwd=tmp, check=True, capture_output=True, timeout=120)
    largest = 0
    for co in glob.glob(so + ".*gfx950"):
        notes = subprocess.run([readelf, "--notes", co], check=True, capture_output=True, text=True, timeout=120).stdout
        for size, name in re.findall(r"\.group_segment_fixed_size:\s+(\d+).*?\.name:\s+(_Z\S+)", notes, re.S):
            if any(k in name for k in kernels):
                largest = max(largest, int(size))
    assert largest > 0
    return largest


def test_solve_plans_fit_lds(plan_test, tmp_path):
    static = _static_lds(str(tmp_path), ("solve_tile_kernel",))
    batch = _static_lds(str(tmp_path), ("batch_solve_kernel", "batch_line_kernel"))
    chunks = _static_lds(str(tmp_path), ("long_forward_kernel", "long_backward_kernel"))
    out = subprocess.run([plan_test, str(static), str(chunks), str(batch)], capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stdout
