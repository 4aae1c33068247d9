"""The choice between caller order and grouping (group_rule.hpp), on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_group_rule_chooses_the_faster(tmp_path):
    exe = str(tmp_path / "group_rule_test")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17",
                    "-I" + os.path.join(ROOT, "bsplineinterpolation_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "group_rule_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
