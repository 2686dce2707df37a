"""The workspace pool on the CPU: pool.hip compiled with tests/hip_stub's
host interface, one case each (pool_cases.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = os.path.join(ROOT, "tests", "hip_stub")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pool") / "pool_cases")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-I", STUB, os.path.join(STUB, "pool_cases.cpp"), "-o",
                    out, "-pthread"], check=True)
    return out


@pytest.mark.parametrize("case", ["renew", "same_handle", "per_thread", "all_of_a_plan", "other_memory", "trim"])
def test_pool(exe, case):
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_all_device_memory_comes_through_the_pool():
    """A hipMalloc elsewhere would fail while the pool holds what it needs."""
    csrc = os.path.join(ROOT, "tom_amd", "csrc")
    for f in sorted(os.listdir(csrc)):
        if f != "pool.hip":
            for line in open(os.path.join(csrc, f)):
                assert "hipMalloc(" not in line.split("//")[0], (f, line)
