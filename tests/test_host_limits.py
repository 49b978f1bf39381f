"""The size limits of mripy_amd/csrc/gn_host_plan.h at sizes too large to run
(tests/host_limits.cpp).  Plain g++; no GPU, no HIP runtime."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_host_limits(tmp_path):
    exe = str(tmp_path / "host_limits")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=undefined", "-fno-sanitize-recover=undefined", "-I",
                        os.path.join(ROOT, "mripy_amd", "csrc"), os.path.join(HERE, "host_limits.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr
