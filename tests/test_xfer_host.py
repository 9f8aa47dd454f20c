"""The transfers between the caller's arrays and the device (orctm_amd/csrc/nh_xfer.cpp), compiled for the host over a
runtime of the harness's own (tests/xfer_host.cpp): what arrives where, and what happens when

* only some of the chunks, or none, can be pinned (``pin``): fewer workers, or the runtime's own copies;
* no thread can be started (``threads``): the caller does all the work;
* the runtime holds the caller's arrays already (``held``): its copies take them as they are;
* an array lies on the device (``device``): no thread of the host touches it;
* others transfer too (``beside``): none waits for another's kernels, nor for another's copies the other way;
* transfers go one after the other (``stage``): they share one set of chunks, both ways;
* an upload is small (``queued``): it is left to the stream, which the caller waits for.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the HIP headers")
    out = str(tmp_path_factory.mktemp("xfer") / "xfer_host")
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-w", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", out, os.path.join(HERE, "xfer_host.cpp")], check=True)
    return out


@pytest.mark.parametrize("check", ["pin", "threads", "held", "device", "beside", "stage", "queued"])
def test_transfer(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr
