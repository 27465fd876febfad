"""The planners of the cell kernels as host code (g++, no device)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pylith_amd", "csrc")


def test_host_memory_running_out_in_a_planner(tmp_path):
    """A failed allocation in one of a planner's threads reaches the planner's caller as an exception."""
    exe = str(tmp_path / "plan_alloc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, os.path.join(ROOT, "tests", "cpp", "plan_alloc.cpp"),
                    os.path.join(CSRC, "plx_plan.cpp"), "-lpthread", "-o", exe], check=True)
    out = subprocess.run([exe, "10"], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.count("reached the caller") == 5
