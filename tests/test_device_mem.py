"""The memory that outlives a handle (device blocks, pinned blocks, staging
buffers with their events) on the CPU: device_mem.cpp and host_copy.cpp built
with g++ under sanitizers against a runtime whose device memory is addresses
only, driven by device_mem_check.cpp: the stated bounds, the retry of a failed
allocation, lists that cannot grow."""
import os
import shutil
import subprocess

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(TESTS), "nido_amd", "csrc")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not found")
    out = str(tmp_path_factory.mktemp("device_mem") / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-fopenmp",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", os.path.join(TESTS, "device_mem_check.cpp"),
                    os.path.join(CSRC, "device_mem.cpp"), os.path.join(CSRC, "host_copy.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("scenario", ["bounded", "retry", "no_memory", "pinned", "staged"])
def test_kept_memory(exe, scenario):
    r = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=60, env=dict(os.environ, OMP_NUM_THREADS="2"))
    assert r.returncode == 0 and "ok" in r.stdout, (r.stdout[-3000:], r.stderr[-3000:])
