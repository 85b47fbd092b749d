"""The device memory pools' bookkeeping (pool.cpp) and the order of forked streams
(fork.hpp) on the CPU: built with stand-ins for the runtime's calls, and the pools
once more under the thread sanitizer."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM", "/opt/rocm")
CASES = ["reuse", "oldest_go", "failing_allocation", "free_without_locks", "per_device", "threads", "forks"]


def build(tmp, *flags):
    exe = os.path.join(tmp, "pool_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-isystem", f"{ROCM}/include",
                    "-I", f"{ROOT}/include", "-I", f"{ROOT}/mxc_amd/csrc/device", *flags, f"{ROOT}/tests/pool_host.cpp",
                    f"{ROOT}/mxc_amd/csrc/device/pool.cpp", "-o", exe, "-pthread"], check=True)
    return exe


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    return build(str(tmp_path_factory.mktemp("pool")))


@pytest.mark.timeout(60)
@pytest.mark.parametrize("case", CASES)
def test_pool(exe, case):
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0, r.stderr


@pytest.mark.timeout(120)
def test_pool_has_no_races(tmp_path):
    exe = build(str(tmp_path), "-fsanitize=" + "thread")
    for case in ("threads", "free_without_locks"):
        r = subprocess.run([exe, case], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
