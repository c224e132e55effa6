"""The order-1 3-D replay leaves a problem to global memory at once where the widest band
of a homogeneous medium comes near its tables in LDS: that estimate, compiled for the
host from the product source, against the band's cells counted one by one."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_band_estimate(tmp_path):
    exe = str(tmp_path / "sfl_band")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-ffp-contract=off", "-w",
           os.path.join(HERE, "native", "sfl_band.hip"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
