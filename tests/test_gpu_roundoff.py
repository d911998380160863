"""Round-off of the FFTs whose column passes end in radix 8, where an inexact sqrt(1/2) shows most: at the top of their
range it stays within the limits' own criterion (Gumbel Z = 28, tests/test_gpu_roe.py)."""
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
