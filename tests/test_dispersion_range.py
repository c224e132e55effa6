"""The queue dispersion kernel takes fp64_ops.h's short quotients and square roots for
columns, periods and velocities that dsp_in_range accepts, where the evaluation says
that its numbers stayed in range.  Built for the host with a fp64_ops.h that
looks at every operand: no accepted evaluation has one outside 2^+-900, and no
earth model, in km or in m, is refused."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "mctomo_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

CHECKED = """
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
extern long fp_bad;
#define FP_HD __host__ __device__ __forceinline__
FP_HD void fp_look(double x)
{
#ifndef __HIP_DEVICE_COMPILE__
    if (x != 0.0 && (fabs(x) <= 0x1p-900 || fabs(x) >= 0x1p900)) fp_bad++;   // (a NaN stays one)
#endif
}
FP_HD double fp_recip(double d) { return 1.0 / d; }
FP_HD double fp_quot(double n, double d, double)
{
    fp_look(n); fp_look(d); fp_look(n / d);
    return n / d;
}
FP_HD double fp_div(double n, double d) { return fp_quot(n, d, 0.0); }
FP_HD double fp_sqrt(double x) { fp_look(x); return sqrt(x); }
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_short_forms_stay_in_range(tmp_path):
    src = tmp_path / "mctomo_amd" / "csrc"
    shutil.copytree(CSRC, src, ignore=shutil.ignore_patterns("*.py", "__pycache__"))
    shutil.copytree(os.path.join(HERE, "..", "include"), tmp_path / "include")
    used = set(re.findall(r"\b(fp_\w+)\(", open(os.path.join(CSRC, "dispersion.hip")).read()))
    assert used <= set(re.findall(r"double (fp_\w+)\(", CHECKED))
    (src / "fp64_ops.h").write_text(CHECKED)
    exe = str(tmp_path / "dltar_range")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-ffp-contract=off", "-w", "-I" + str(src),
           os.path.join(HERE, "native", "dltar_range.hip"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe, "200000"], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
