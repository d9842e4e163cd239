"""CPU check of the way fields take to the host (csrc/fetch.hpp).

fetch_check.cpp plays the HIP runtime: a copy into pinned memory runs no
earlier than the wait that promises it.  Contexts share the lanes that the
first has pinned, never two at a time, and where pinning fails contexts are
made and fields arrive all the same.  Values are compared one by one at the
sizes where the way changes (around pieces of 1 MiB and the size from which
four threads take a part each), FP32 and FP64, and a failing copy is reported.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "komegafoulingmodel_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_fields_arrive_whole_through_shared_lanes(tmp_path):
    exe = tmp_path / "fetch_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    "-I", CSRC, os.path.join(HERE, "fetch_check.cpp"), "-o", str(exe), "-pthread"], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(res.stdout[-2000:])
    assert res.returncode == 0
