"""The wave lines of every listed box length, on the host:
tests/wave_lines_host.hip includes the headers of the kernels and is built here
with hipcc."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_wave_line_layouts(tmp_path):
    cc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(cc):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "wave_lines")
    r = subprocess.run([cc, "-O1", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", os.path.join(HERE, "wave_lines_host.hip"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert "lengths 45 failures 0" in r.stdout
