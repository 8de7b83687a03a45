"""Band-limit, template and aperture ranges, their columns and the
nearest-pixel index (tests/host/ranges_check.cpp): the bisections against a
test of every pixel, 400 grids, compiled with g++ as the library's host unit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = [os.path.join(ROOT, "tests", "host", "ranges_check.cpp"),
       os.path.join(ROOT, "ms-stem-fem_amd", "csrc", "msf_host.cpp")]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_ranges_equal_a_test_of_every_pixel(tmp_path):
    exe = str(tmp_path / "ranges_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fno-fast-math", "-pthread",
                    "-Wall", *SRC, "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0
    assert r.stdout.strip() == "ranges 0 columns 0 indices 0 whole rows 1"
