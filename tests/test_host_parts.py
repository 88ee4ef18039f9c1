"""How the host pool cuts a range into parts, compiled on the CPU with g++
(tests/host_parts_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_no_more_parts_than_threads(tmp_path):
    exe = tmp_path / "host_parts_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-o", str(exe),
                    os.path.join(ROOT, "tests", "host_parts_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout
