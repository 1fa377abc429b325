"""Pools of device blocks: their rules on the CPU, against a device of counted bytes (tests/c/pool.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "r-scape_amd", "csrc")


def test_pool_rules(tmp_path):
    """Reuse by size class, bounds, release with the pool and on request, release by all pools when
    the device is full, host memory that runs out at any allocation, eight threads on two pools."""
    exe = str(tmp_path / "pool")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           os.path.join(ROOT, "tests", "c", "pool.cpp"), "-x", "c++", os.path.join(CSRC, "rsg_pool.hip"),
                           "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.splitlines()[-1] == "threads ok", r.stdout + r.stderr
