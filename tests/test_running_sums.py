"""Running sums of block probabilities on the host (tests/native/running_sums_test.cpp), built with
g++ under AddressSanitizer and UndefinedBehaviorSanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-fno-omit-frame-pointer"]


def test_running_sums(tmp_path):
    hip_inc = "/opt/rocm/include"
    if not os.path.isdir(os.path.join(hip_inc, "hip")):
        pytest.skip("HIP headers not installed")
    exe = str(tmp_path / "running_sums_test")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I" + hip_inc] + SAN +
                   [os.path.join(HERE, "native", "running_sums_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "running sums ok" in out.stdout, out.stdout[-2000:] + out.stderr[-4000:]
