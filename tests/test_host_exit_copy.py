"""The copy of exit waves to the caller (tests/host/exit_copy_check.cpp): the
library's unit on a stand-in for the runtime that copies as late as it may,
with and without pinned memory, also under ThreadSanitizer (host code only)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
SRC = [os.path.join(ROOT, "tests", "host", "exit_copy_check.cpp"),
       os.path.join(ROOT, "ms-stem-fem_amd", "csrc", "msf_exit.cpp")]


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(ROCM + "/include/hip"),
                    reason="g++ or the HIP headers not available")
@pytest.mark.parametrize("san", ["", "thread"])
def test_exit_waves_arrive_whole(tmp_path, san):
    exe = str(tmp_path / "exit_copy_check")
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-pthread", "-D__HIP_PLATFORM_AMD__",
           f"-I{ROCM}/include", *SRC, "-o", exe]
    if san:
        cmd.insert(1, f"-fsanitize={san}")
    subprocess.run(cmd, check=True, timeout=300)
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=1")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0, r.stderr[-4000:]
    assert r.stdout.strip() == "plain 0 both 0 flight 0 silent 0 kept 1 left 0 refused 0"
