"""The FP64 quotients of the kernels (hamr_arith.h) at the ends of the exponent range,
on the host (tests/arith/check_div_range.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hamr_gamma_wind_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_quotients_at_the_ends_of_the_range(tmp_path):
    exe = str(tmp_path / "check_div_range")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-I" + CSRC,
                        os.path.join(HERE, "arith", "check_div_range.cpp"), "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
