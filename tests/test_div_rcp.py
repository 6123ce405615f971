"""The exact kernels' quotient by a rounded reciprocal (div_by_rcp in feriphys_amd/csrc/exact_ops.hpp) equals
the division: on every pair of significands whose quotient is close enough to a midpoint of two floats to be
misrounded (tests/native/div_rcp_check.cpp derives them) and on 2^27 random pairs over the range of exponents
that the callers allow."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_quotient_by_reciprocal_is_the_division(tmp_path):
    exe = str(tmp_path / "div_rcp_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-fno-fast-math", "-fopenmp",
                    os.path.join(HERE, "native", "div_rcp_check.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["33555480", "0", str(1 << 27), "0"]
