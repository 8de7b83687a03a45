"""Kept sets that are not disks in FFT order are reported as such
(tests/host/ranges_refused.cpp), compiled with g++ as the library's host
unit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = [os.path.join(ROOT, "tests", "host", "ranges_refused.cpp"),
       os.path.join(ROOT, "ms-stem-fem_amd", "csrc", "msf_host.cpp")]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_sets_that_are_no_disks_are_reported(tmp_path):
    exe = str(tmp_path / "ranges_refused")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fno-fast-math", "-pthread",
                    "-Wall", *SRC, "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0
    assert r.stdout.strip() == "refused 0 accepted 0"
