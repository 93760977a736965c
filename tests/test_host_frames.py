"""The host side of a frame on a stand-in device: tests/native/host_frame_check.cpp
compiles blend2d_amd/csrc/context.cpp with functions in place of the HIP calls
and kernel launches, so that counts, the memory left and the current device can
be chosen.  Nothing is rendered."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP_INCLUDE = "/opt/rocm/include"
CASES = ["enough", "more_segments", "more_clip_items", "tight_device", "too_tight", "counts_differ", "other_device",
         "schedules"]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists(os.path.join(HIP_INCLUDE, "hip", "hip_runtime.h")):
        pytest.skip("g++ or the HIP headers are missing")
    out = tmp_path_factory.mktemp("host") / "check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + HIP_INCLUDE, "-o", str(out),
                    os.path.join(ROOT, "tests", "native", "host_frame_check.cpp"),
                    os.path.join(ROOT, "blend2d_amd", "csrc", "style.cpp"), "-lpthread"], check=True)
    return str(out)


@pytest.mark.parametrize("case", CASES)
def test_case(exe, case):
    res = subprocess.run([exe, case], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
