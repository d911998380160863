"""What was read back of a residue packed on the device is believed only when two heads and an independent sum of the
digits agree (gpuowl_amd/csrc/pack.h), checked on the CPU: no single wrong bit in a head, in the words or in the
packing passes, and a head that was never written is not a zero residue."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not installed")
def test_wrong_reads_are_not_believed(tmp_path):
    exe = tmp_path / "pack_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "gpuowl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "pack_check.cpp"), "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout
