"""Host-side check of log_pos and div_normal (botorch_amd/csrc/bta_common.h): within
one unit in the last place of the long double results, compiled with hipcc and run
on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_log_pos_within_one_ulp(tmp_path):
    exe = tmp_path / "log_pos_check"
    src = os.path.join(HERE, "native", "log_pos_check.hip")
    subprocess.run([HIPCC, "-O2", "--offload-arch=gfx950", "-std=c++17", src, "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
