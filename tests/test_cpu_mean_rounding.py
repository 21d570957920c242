"""The fast march's rounding correction stays a rounding for any finite density,
subnormal ones included (host build; no GPU needed)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_correction_is_a_rounding(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = tmp_path / "mean_rounding_check"
    src = os.path.join(HERE, "native", "mean_rounding_check.hip")
    r = subprocess.run([hipcc, "-O2", "-std=c++17", "-ffp-contract=off", src, "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
