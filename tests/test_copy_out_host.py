"""The staged copies to the host (HostStaging in mf-lbm-cuda_amd/csrc/copy_out.h) with the HIP calls
replaced by host ones, on the CPU: contents at the sizes where chunks and slots change, the order
of its locks, the thread that makes the HIP calls, the destinations that need no staging, the copy
that makes the slots, errors, and copies from several threads."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mf-lbm-cuda_amd", "csrc")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("copy_out") / "copy_out_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC,
                    os.path.join(HERE, "copy_out_check.cpp"), "-o", out], check=True, timeout=120)
    return out


@pytest.mark.parametrize("check", ["contents", "order", "calls", "destinations", "worth", "errors", "threads", "waits"])
def test_staged_copy(harness, check):
    """exit status 1: it did not hold, 3: it did not end"""
    assert subprocess.run([harness, check], timeout=60).returncode == 0
