"""The adjoint's reverse parabola (`para_vjp`, hamr_adjoint.h) equals the
transposed Jacobian (`para_jacobian`) on 1e6 stencils: random, near-linear,
spiked and with ties (para, GPU_interp.h:60-111)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hamr_gamma_wind_amd", "csrc")
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_reverse_parabola_equals_transposed_jacobian(tmp_path):
    exe = str(tmp_path / "check_ppm_vjp")
    cmd = [HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "-I" + CSRC, "-x", "hip", "--offload-arch=gfx950",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           os.path.join(HERE, "adjoint_ppm", "check_ppm_vjp.cpp"), "-o", exe]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
