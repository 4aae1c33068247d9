"""Factors with settled rows copied (setup.cpp) against the elimination of
every entry, on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bsplineinterpolation_amd", "csrc")


def test_factors_equal_plain_elimination(tmp_path):
    exe = str(tmp_path / "factor_test")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-ffp-contract=off", "-I" + CSRC,
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", "factor_test.cpp"),
                    os.path.join(CSRC, "setup.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stdout
