"""Host-side helpers of the library's sources, compiled into small programs of
their own (tests/cpp/*_check.cpp) and run without a GPU."""
import os
import shutil
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is not installed")
@pytest.mark.parametrize("name", ["parts_check", "lanes_check", "fft_check"])
def test_host_check(name, tmp_path):
    exe = str(tmp_path / name)
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", os.path.join(CPP, name + ".cpp"), "-o", exe]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout.strip() == "ok", (res.returncode, res.stdout,
                                                                res.stderr)
