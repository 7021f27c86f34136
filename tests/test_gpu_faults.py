"""Allocations refused from the host (tests/cpp/faults.cpp): what a call falls
back to, and what it leaves."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def faults(tmp_path_factory):
    import exafmm_amd as F
    exe, libdir = str(tmp_path_factory.mktemp("faults") / "faults"), os.path.dirname(F.LIB_PATH)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", "faults.cpp"), "-o", exe,
                    "-L", libdir, "-lexafmm_amd", "-Wl,-rpath," + libdir, "-L", "/opt/rocm/lib", "-lamdhip64",
                    "-Wl,-rpath,/opt/rocm/lib", "-ldl"], check=True)

    def run(what):
        out = subprocess.run([exe, what], capture_output=True, text=True, timeout=100)
        print(out.stdout, flush=True)
        assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout + out.stderr
    return run


def test_groups_on_the_host(faults):
    faults("groups")


def test_system_kept_when_the_next_fails(faults):
    faults("kept")
