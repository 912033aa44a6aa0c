"""The FP64 quotients and powers the kernels form on the device (hamr_arith.h)
against IEEE division and a 113-bit power, on the host (tests/arith/check_arith.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hamr_gamma_wind_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_quotients_and_powers(tmp_path):
    exe = str(tmp_path / "check_arith")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-I" + CSRC,
                        os.path.join(HERE, "arith", "check_arith.cpp"), "-o", exe, "-lquadmath"],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
