"""The autotuner's candidates for batches that take the one-launch slice loop
(tests/host/tune_loop_check.cpp), compiled with g++ as the library's host
unit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = [os.path.join(ROOT, "tests", "host", "tune_loop_check.cpp"),
       os.path.join(ROOT, "ms-stem-fem_amd", "csrc", "msf_host.cpp")]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_one_candidate_per_slice_loop(tmp_path):
    exe = str(tmp_path / "tune_loop_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fno-fast-math", "-pthread",
                    "-Wall", *SRC, "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0
    assert r.stdout.strip() == "loop 0 tiles 0 loops 1"
