"""The split W x H and line block R of a job that runs alone, at the edges of the rule that chooses them, against GMP:
the longest columns of one width, the largest FFT with two-line blocks, words too short for the carries of two-line
blocks, and the last exponents below an FFT's limit."""
import sys

import pytest

import gpuowl_amd as owl
import oracle
from gpuowl_amd import workloads

pytestmark = pytest.mark.gpu

# (spec, bits per word or None for an exponent at the FFT's limit, W, H, R)
CASES = [("256:2:256", 9, 256, 512, 2), ("256:8:256", 9, 256, 2048, 2), ("256:9:256", 9, 512, 1152, 2),
         ("256:11:512", 9, 1024, 1408, 2), ("1K:6:256", 9, 1024, 1536, 4), ("1K:16:256", 9, 1024, 4096, 4),
         ("256:8:256", 5, 256, 2048, 2), ("256:8:256", 4, 256, 2048, 8), ("256:3:256", None, 256, 768, 4),
         ("256:9:256", None, 256, 2304, 8)]


@pytest.mark.parametrize("spec,bits,W,H,R", CASES)
def test_split_of_a_job_alone(spec, bits, W, H, R):
    _, N, limit = owl.best_fit(1000, spec)
    E = workloads.primes_from(bits * N if bits else limit - 1000, 1)[0]
    print("CASE", spec, E, file=sys.stderr, flush=True)
    with owl.Gpu(E, spec) as g:
        assert (g.W, g.H, g.R) == (W, H, R) and g.row_kernel == f"rowx{W}r{R}" and g.col_kernel.startswith(f"colx{H}")
        r, _ = g.prp(40, block_size=20, check_step=20)
        assert r.res64 == oracle.gmp_res64(E, 40, 40)[0] and r.nErrors == 0 and r.maxRoe < 0.45
