"""Host passes over neurons on several threads (compiled with g++): running
out of memory while they start neither ends the process nor skips a part."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_parts_out_of_memory(tmp_path):
    exe = tmp_path / "parts_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I",
                    os.path.join(ROOT, "digital_twin_brain-open_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "parts_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
