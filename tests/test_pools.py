"""Pools of memory and streams (csrc/memory_pool.hip) and the rows of a matrix (csrc/float_rows.hip) on the CPU,
over a stand-in for the HIP runtime with several devices."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "arboretum_amd", "csrc")


def _build(out, check, sources):
    native = os.path.join(HERE, "native")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                           "-o", out, "-x", "c++"] + [os.path.join(CSRC, s) for s in sources] +
                          [os.path.join(native, "fake_hip.cpp"), os.path.join(native, check)])


def _run(program, check):
    r = subprocess.run([program, check], stdout=subprocess.PIPE, timeout=60)
    assert r.returncode == 0, r.stdout.decode()


@pytest.fixture(scope="module")
def pools(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pools") / "check_pools")
    _build(out, "check_pools.cpp", ["memory_pool.hip"])
    return out


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rows") / "check_rows")
    _build(out, "check_rows.cpp", ["memory_pool.hip", "float_rows.hip", "staging.hip", "parallel.cpp"])
    return out


@pytest.mark.parametrize("check", ["other_device", "threads", "bounds", "release"])
def test_pool(pools, check):
    _run(pools, check)


@pytest.mark.parametrize("check", ["other_device", "places"])
def test_rows(rows, check):
    _run(rows, check)
