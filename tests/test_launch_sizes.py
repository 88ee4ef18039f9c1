"""What the launches are sized by, checked on the host: tests/launch_check.cpp
compiled with g++ against ngap_amd/csrc/kernels.h (no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_launch_sizes(tmp_path):
    exe = tmp_path / "launch_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-o", str(exe),
                    os.path.join(ROOT, "tests", "launch_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout
