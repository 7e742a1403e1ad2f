"""Error paths of the device library's host code, on the CPU: test programs (host_failures/) that
link the library and define the HIP calls themselves, so that a launch or an allocation can be
made to fail at a chosen place."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "host_failures")
PKG = os.path.join(ROOT, "cpu-ipc_amd")


@pytest.mark.parametrize("program", ["solve", "read_arrays"])
def test_failure(program, tmp_path):
    exe = str(tmp_path / program)
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-Wno-unused-result",
                        "-I", os.path.join(PKG, "csrc"), os.path.join(HERE, program + ".cpp"), "-o", exe, "-rdynamic",
                        "-L", PKG, "-l:libcipc_gpu.so", "-Wl,-rpath," + PKG], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
