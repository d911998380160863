"""Round-off of the FFTs whose column passes end in radix 8, where an inexact sqrt(1/2) shows most: at the top of their
range it stays within the limits' own criterion (Gumbel Z = 28, tests/test_gpu_roe.py). And round-off of the split that a job
alone takes, at the last exponents that have it (0.997 of an FFT's limit): below what the same exponents had in the
reference's split before there was one."""
import sys

import pytest

import gpuowl_amd as owl
from gpuowl_amd import workloads

pytestmark = pytest.mark.gpu


def prev_prime(n):
    while not workloads.is_prime(n):
        n -= 1
    return n


def measure(E, spec):
    with owl.Gpu(E, spec) as g:
        r = g.measure_roe(10000, 50)
        r["split"] = (g.W, g.H, g.R)
    print(f"ROE {spec} E={E} {r}", file=sys.stderr, flush=True)
    assert r["n"] == 10000
    return r


# 256 x 1024 twice, 256 x 1280, 256 x 2048 and 1024 x 1280
@pytest.mark.parametrize("spec", ["256:4:256:101", "256:2:512:202", "256:5:256:202", "256:8:256:202", "1K:5:256:202"])
def test_round_off_at_the_limit(spec):
    r = measure(prev_prime(owl.best_fit(1000, spec)[2]), spec)
    assert r["z"] >= 28 and r["max"] < 0.4, r


# (spec, W, H, R, mean largest round-off over 20,000 squarings in the reference's split with the pass before k_colx kept its
# butterflies in registers). The mean of 10,000 squarings has a standard error of 0.07%.
ALONE = [("256:4:256:101", 256, 1024, 2, 0.17804), ("256:9:256:101", 512, 1152, 2, 0.15832),
         ("256:10:256:202", 512, 1280, 2, 0.17472), ("1K:3:256:101", 512, 1536, 2, 0.14289),
         ("1K:4:256:202", 512, 2048, 2, 0.15928), ("256:16:256:202", 512, 2048, 2, 0.18561),
         ("256:11:512:202", 1024, 1408, 2, 0.17028)]


@pytest.mark.parametrize("spec,W,H,R,before", ALONE)
def test_round_off_of_the_split_for_jobs_alone(spec, W, H, R, before):
    limit = owl.best_fit(1000, spec)[2]
    r = measure(prev_prime(int(0.997 * limit)), spec)
    assert r["split"] == (W, H, R)
    assert r["z"] >= 28 and r["mean"] <= before, r
    at_limit = measure(prev_prime(limit), spec)
    assert at_limit["split"] != (W, H, R) and r["mean"] <= at_limit["mean"], at_limit
