"""Planning time of gate programs and Pauli sums over long inputs, on the host
(tests/native/plan_scaling_test.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hiqsimulator_amd", "csrc")


def test_planning_scales(tmp_path):
    hip_inc = "/opt/rocm/include"
    if not os.path.isdir(os.path.join(hip_inc, "hip")):
        pytest.skip("HIP headers not installed")
    exe = str(tmp_path / "plan_scaling_test")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I" + hip_inc] +
                   [os.path.join(CSRC, s) for s in ("gate_prog.cpp", "pauli_prog.cpp")] +
                   [os.path.join(HERE, "native", "plan_scaling_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "planning scales" in out.stdout, out.stdout + out.stderr[-4000:]
