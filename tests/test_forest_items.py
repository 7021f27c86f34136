"""M2L work items of merged plans (tests/cpp/forest_items_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_items_of_a_forest(tmp_path):
    csrc, exe = os.path.join(ROOT, "exafmm-beta_amd", "csrc"), str(tmp_path / "forest_items_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", csrc,
                    os.path.join(ROOT, "tests", "cpp", "forest_items_check.cpp"), os.path.join(csrc, "fmm_host.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout
