"""Which way gate lists go (gate_list_cost, gate_route), on the host: tests/native/gate_route_test.cpp,
built with g++ under AddressSanitizer and UndefinedBehaviorSanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hiqsimulator_amd", "csrc")
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-fno-omit-frame-pointer"]


def test_gate_routes(tmp_path):
    hip_inc = "/opt/rocm/include"
    if not os.path.isdir(os.path.join(hip_inc, "hip")):
        pytest.skip("HIP headers not installed")
    exe = str(tmp_path / "gate_route_test")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__", "-I" + hip_inc] + SAN +
                   [os.path.join(CSRC, "gate_prog.cpp"), os.path.join(HERE, "native", "gate_route_test.cpp"), "-o", exe],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "gate routes ok" in out.stdout, out.stdout[-2000:] + out.stderr[-4000:]
