"""Job tables that are uploaded only when they changed (mpsq_buffers.h):
native/arena_check.cpp runs the real header on the host, over a stand-in for
the HIP runtime, with allocations that fail between a table's change and its
upload."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_device_tables_follow_the_host(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not installed")
    exe = str(tmp_path / "arena_check")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "mp_tools_amd", "csrc"),
                           os.path.join(ROOT, "tests", "native", "arena_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
