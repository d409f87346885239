"""The engine's host code over a stand-in for the HIP runtime (tests/native/fake_hip.hpp), built
with g++ under AddressSanitizer and UndefinedBehaviorSanitizer: allocations and launches that fail
on the way leave the state and the queue as a caller who goes on needs them."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hiqsimulator_amd", "csrc")
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-fno-omit-frame-pointer"]


@pytest.mark.parametrize("unit,said", [("gate_failure", "gate failures ok"),
                                       ("evolve_failure", "evolution failures ok")])
def test_failures_on_the_way(tmp_path, unit, said):
    hip_inc = "/opt/rocm/include"
    if not os.path.isdir(os.path.join(hip_inc, "hip")):
        pytest.skip("HIP headers not installed")
    exe = str(tmp_path / (unit + "_test"))
    srcs = [os.path.join(CSRC, s) for s in ("engine.cpp", "sched.cpp", "gate_prog.cpp", "pauli_prog.cpp")]
    # kernels that no test reaches stay unresolved
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + hip_inc, "-no-pie",
                    "-Wl,--unresolved-symbols=ignore-all"] + SAN +
                   srcs + [os.path.join(HERE, "native", unit + "_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert out.returncode == 0 and said in out.stdout, out.stdout[-2000:] + out.stderr[-4000:]
