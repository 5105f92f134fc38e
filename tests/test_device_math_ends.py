"""Host-side check of div_by and log_pos (botorch_amd/csrc/bta_common.h) at the ends of
their ranges, compiled with hipcc and run on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("what", ["div", "log"])
def test_quotients_and_logs_at_the_ends_of_their_ranges(tmp_path, what):
    exe = tmp_path / "div_log_ends_check"
    src = os.path.join(HERE, "native", "div_log_ends_check.hip")
    subprocess.run([HIPCC, "-O2", "--offload-arch=gfx950", "-std=c++17", src, "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)
    r = subprocess.run([str(exe), what], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
