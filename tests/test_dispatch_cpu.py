"""The host's choices of forms, teams and slices on the CPU, under AddressSanitizer
and UBSan (tests/cpu_checks/dispatch_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_dispatch_under_sanitizers(tmp_path):
    exe = str(tmp_path / "dispatch_check")
    src = os.path.join(HERE, "cpu_checks", "dispatch_check.cpp")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                           "-fno-sanitize-recover=all", "-o", exe, src])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "dispatch checks passed" in out.stdout
