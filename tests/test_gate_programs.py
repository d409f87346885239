"""Gate programs and Pauli sums on the host: the unit splitter, the planners and the compiler
against plain interpreters of the compiled records (tests/native/
gate_prog_test.cpp, pauli_prog_test.cpp), built with g++ under AddressSanitizer and
UndefinedBehaviorSanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hiqsimulator_amd", "csrc")
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-fno-omit-frame-pointer"]


@pytest.mark.parametrize("unit,said", [("gate_prog", "gate programs ok"), ("pauli_prog", "pauli plans ok")])
def test_programs_under_sanitizers(tmp_path, unit, said):
    hip_inc = "/opt/rocm/include"
    if not os.path.isdir(os.path.join(hip_inc, "hip")):
        pytest.skip("HIP headers not installed")
    exe = str(tmp_path / (unit + "_test"))
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I" + hip_inc] + SAN +
                   [os.path.join(CSRC, unit + ".cpp"), os.path.join(HERE, "native", unit + "_test.cpp"), "-o", exe],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert out.returncode == 0 and said in out.stdout, out.stdout[-2000:] + out.stderr[-4000:]
