"""P2M's sums over a leaf's groups of lanes stay inside their buffer: walked on
the host for every order and both forms of the kernel (tests/cpp/p2m_lanes_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lanes_read_their_own_leaf(tmp_path):
    exe = str(tmp_path / "p2m_lanes_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "exafmm-beta_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "p2m_lanes_check.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
