"""The channel sums of the adaptive search, thread by thread on the CPU
(tests/cpp/test_opt_decide.cpp): for every grid size no thread stores past the
scratch the launch asks for."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_sums_stay_in_their_scratch(tmp_path):
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "beamform_project_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_opt_decide.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "OK" in r.stdout, r.stdout + r.stderr
