"""Spread tile shapes: every shape the library accepts fits the kernels it
runs on (native/tiles_check.cpp, compiled for the host), and one that does not
is refused."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_accepted_tiles_fit_their_kernels(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not installed")
    exe = str(tmp_path / "tiles_check")
    subprocess.check_call([hipcc, "-O2", "-std=c++17", "--offload-arch=gfx950", "-I",
                           os.path.join(ROOT, "mp_tools_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                           os.path.join(ROOT, "tests", "native", "tiles_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr


@pytest.mark.gpu
def test_odd_tile_beyond_the_complex_kernel(gpu_lib):
    """25 rows of 512 cells: no pairs for the real kernel, and more rows than
    the complex one transforms."""
    from mp_tools_amd._lib import MpsqError
    from mp_tools_amd.sqw import SqwEngine
    with pytest.raises(MpsqError):
        SqwEngine(3, (256, 50, 50), (100,), precision="fp32", tile_by=5, tile_bz=5)
    SqwEngine(3, (256, 50, 50), (100,), precision="fp32", tile_by=5, tile_bz=4)
