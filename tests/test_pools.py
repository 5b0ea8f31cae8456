"""Pools of memory and streams (csrc/memory_pool.hip) on the CPU, over a stand-in for the HIP runtime with
several devices."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "arboretum_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pools") / "check_pools")
    native = os.path.join(HERE, "native")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                           "-o", out, "-x", "c++", os.path.join(CSRC, "memory_pool.hip"),
                           os.path.join(native, "fake_hip.cpp"), os.path.join(native, "check_pools.cpp")])
    return out


@pytest.mark.parametrize("check", ["other_device", "threads", "bounds", "release"])
def test_pool(program, check):
    r = subprocess.run([program, check], stdout=subprocess.PIPE, timeout=60)
    assert r.returncode == 0, r.stdout.decode()
