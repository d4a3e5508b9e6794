"""The pinned memory of a call: it keeps the no-allocation promise of
dtb_run_noalloc (it throws instead of growing), and the state goes through it
in pieces where device memory is short.  Programs compiled with g++ against
the library's own headers."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def run_native(dtb, tmp_path, name):
    exe, lib, rocm = tmp_path / name, os.path.dirname(dtb.LIB_PATH), "/opt/rocm"
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "digital_twin_brain-open_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", name + ".cpp"), "-L", lib, "-ldtb",
                    "-L", os.path.join(rocm, "lib"), "-lamdhip64", "-Wl,-rpath," + lib,
                    "-Wl,-rpath," + os.path.join(rocm, "lib"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr


def test_no_pinned_allocation_under_noalloc(dtb, tmp_path):
    run_native(dtb, tmp_path, "stage_check")


@pytest.mark.gpu
def test_state_without_device_memory(dtb, gpu, tmp_path):
    run_native(dtb, tmp_path, "state_check")
