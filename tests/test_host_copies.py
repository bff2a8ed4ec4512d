"""Host paths of libmmsim whose calls into HIP fail one after the other, on the CPU.

``host_copies.cpp`` is a program with a HIP runtime of its own, linked with the built library: a copy from or to host memory
happens when its stream is waited for, the n-th call that can fail does.  For every n no memory may go while a copy still
needs it and no device memory may stay behind, and a batch for lanes at their own pace that gets no memory for its further
tables has to become one for another loop."""
import os
import shutil
import subprocess

import pytest

from mms_amd import _lib

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"), reason="needs g++ and HIP's headers")
def test_no_copy_outlives_its_host_memory_whatever_fails(tmp_path):
    exe, libs = str(tmp_path / "host_copies"), os.path.dirname(_lib.LIB_PATH)
    cmd = ["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", os.path.join(HERE, "host_copies.cpp"), "-rdynamic",
           "-pthread", _lib.LIB_PATH, "-Wl,-rpath," + libs, "-Wl,--allow-shlib-undefined", "-o", exe]
    built = subprocess.run(cmd, capture_output=True, text=True)
    assert built.returncode == 0, built.stderr
    proc = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0 and proc.stdout.endswith("ok\n"), proc.stdout + proc.stderr
