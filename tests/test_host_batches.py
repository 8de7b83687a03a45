"""The split of a run's positions into batches (tests/host/batches_check.cpp):
every position count up to 1024 on seven grids, compiled with g++ as the
library's host unit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = [os.path.join(ROOT, "tests", "host", "batches_check.cpp"),
       os.path.join(ROOT, "ms-stem-fem_amd", "csrc", "msf_host.cpp")]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_two_chains_share_an_even_number_of_like_batches(tmp_path):
    exe = str(tmp_path / "batches_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fno-fast-math", "-pthread",
                    "-Wall", *SRC, "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0
    assert r.stdout.strip() == "cover 0 room 0 odd 0 uneven 0 changed 0 fired 1"
