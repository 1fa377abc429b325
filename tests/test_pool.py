"""Pools of device blocks: their rules on the CPU, against a device of counted bytes (tests/c/pool.cpp)."""
import glob
import os
import re
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


def test_every_device_allocation_reclaims_idle_blocks():
    """What the pools keep must not make another allocation of the library fail: device memory is
    allocated through rsg_dev_malloc (pressure case above) and nowhere else."""
    direct = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        if os.path.basename(path) == "rsg_pool.hip":
            continue
        for n, line in enumerate(open(path), 1):
            if re.search(r"\bhip(Ext|Pitched)?Malloc(WithFlags|Managed|Pitch|Async)?\s*\(", line.split("//")[0]):
                direct.append("%s:%d" % (os.path.basename(path), n))
    assert not direct, direct
