"""The small DFTs of every pass, on the CPU from the kernel header itself (tests/small_dft_check.cpp): the error of an output
may not have a part that always points the same way, as sqrt(1/2) and sqrt(3)/2 rounded to double give it (0.31 of 2^-53
for radix 8, 0.52 for radix 12): from stage to stage such errors add up where rounding errors average out."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
# Radices whose roots are rational but for sqrt(1/2) and sqrt(3)/2 have nothing left but the noise of 100,000 samples: an rms
# error below 1.1 over sqrt(100,000) per output, 0.0035, of which 0.02 is almost six times. The others keep the rounding of their own
# constants, at most half of 2^-53 each and of both signs: below 0.15.
EXACT, OTHERS = 0.02, 0.15


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_small_dfts_have_no_systematic_error(tmp_path):
    exe = tmp_path / "small_dft_check"
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-mfma", "-ffp-contract=fast",
                    "-I", os.path.join(ROOT, "gpuowl_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "small_dft_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=300).stdout
    rows = [line.split() for line in out.splitlines()]
    assert [(int(r[0]), int(r[1])) for r in rows] == [(R, i) for R in range(2, 17) for i in (0, 1)]
    for radix, inverse, rms, gain in rows:
        assert float(rms) < 1.25, (radix, inverse)
        assert float(gain) < (EXACT if int(radix) in (2, 3, 4, 6, 8, 12) else OTHERS), (radix, inverse, gain)
