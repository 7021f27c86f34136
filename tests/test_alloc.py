"""Out of device memory: what the plan builders keep for later is given back
before an allocation fails (tests/cpp/alloc_check.cpp, on a made-up device)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_idle_scratch_makes_room(tmp_path):
    import exafmm_amd as F
    exe, libdir = str(tmp_path / "alloc_check"), os.path.dirname(F.LIB_PATH)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                    os.path.join(ROOT, "exafmm-beta_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "alloc_check.cpp"),
                    "-o", exe, "-L", libdir, "-lexafmm_amd", "-Wl,-rpath," + libdir], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
