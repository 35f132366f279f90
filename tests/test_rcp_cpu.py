"""The Newton step of the box tests' reciprocals (luxcore_amd/csrc/lrh_rcp.h):
over every mantissa, from 1/d itself and the floats on either side, it gives
the correctly rounded 1/d, but for single mantissas from a neighbour that is
more than an ulp from 1/d (33 of 25 million; the device's estimates, which are
within an ulp, meet none of them)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("rcp") / "rcp_check"
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17", "-Wall", "-o", str(out),
                    os.path.join(ROOT, "tests", "native", "rcp_check.cpp")], check=True, timeout=180)
    return out


# from the clamp's 1e-20 to the 1e30 above which components are divided
@pytest.mark.parametrize("exponent", [-66, 0, 1, 98])
def test_step_rounds_correctly(exe, exponent):
    tried, differ = map(int, subprocess.run([str(exe), str(exponent), "1"], capture_output=True, text=True, timeout=120,
                                            check=True).stdout.split())
    assert tried == 3 << 23
    assert differ <= 33
    assert int(subprocess.run([str(exe), str(exponent), "0"], capture_output=True, text=True, timeout=120,
                              check=True).stdout.split()[1]) == 0
