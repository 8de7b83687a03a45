"""The autotuner's candidate launch shapes (tests/host/tune_check.cpp), compiled
with g++ as the library's host unit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = [os.path.join(ROOT, "tests", "host", "tune_check.cpp"),
       os.path.join(ROOT, "ms-stem-fem_amd", "csrc", "msf_host.cpp")]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_candidates_hold_the_rule(tmp_path):
    exe = str(tmp_path / "tune_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fno-fast-math", "-pthread",
                    "-Wall", *SRC, "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0
    assert r.stdout.strip() == "rule 0 twice 0 tiles 0 one batch 0 fused 0"
