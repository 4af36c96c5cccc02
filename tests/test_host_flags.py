"""The pool of status slots in pinned host memory
(torchproteinlibrary_amd/csrc/host_flags.h), compiled for the host: a slot goes
back only after the wait for its stream, also when a launch fails."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_slots_after_failures(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    if shutil.which("g++") is None or not os.path.isdir(os.path.join(rocm, "include", "hip")):
        pytest.skip("no host C++ compiler or no HIP headers")
    exe = str(tmp_path / "host_flags")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__=1", "-isystem",
                           os.path.join(rocm, "include"), "-I", os.path.join(ROOT, "torchproteinlibrary_amd", "csrc"),
                           os.path.join(ROOT, "tests", "host_flags_host.cpp"), "-o", exe])
    assert subprocess.run([exe], timeout=60).returncode == 0
