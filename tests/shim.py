"""Runs a piece of Python in a child process whose HIP calls pass hip_shim.cpp
first: the code finds the shim's controls as `shim`, the package as `na`."""
import os
import subprocess
import sys

TESTS = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, sys
sys.path[:0] = [{root!r}, {tests!r}]
shim = ctypes.CDLL({lib!r}, ctypes.RTLD_GLOBAL)
import nido_amd as na
path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln)
assert shim.shim_init(path.encode()) == 0
"""


def run_with_shim(code, tmp_path, timeout=100):
    lib = str(tmp_path / "hip_shim.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(TESTS, "hip_shim.cpp"), "-o", lib, "-ldl"], check=True)
    prelude = PRELUDE.format(root=os.path.dirname(TESTS), tests=TESTS, lib=lib)
    r = subprocess.run([sys.executable, "-c", prelude + code], capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    return r.stdout
