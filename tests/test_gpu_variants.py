"""The squaring's passes in the variants a launch chooses by its number of jobs and the size of their
states (complex or split exchanges, plain or non-temporal accesses), against GMP. One shape's batch
sizes lie on either side of each limit: the number of column pairs that gives every CU two groups, and
56 MB and 256 MB of states."""
import sys

import pytest

import gpuowl_amd as owl
import oracle
from gpuowl_amd import workloads

pytestmark = pytest.mark.gpu

# (spec, width, line block, jobs)
CASES = [("256:2:256", 256, 4, 1), ("256:9:256", 256, 8, 1), ("256:9:256", 256, 8, 4), ("256:9:256", 256, 8, 8),
         ("256:9:256", 256, 8, 29), ("1K:6:256", 1024, 4, 1), ("1K:6:256", 1024, 4, 3), ("256:9:512", 512, 4, 2),
         ("1K:15:256", 1024, 4, 1)]


@pytest.mark.parametrize("spec,width,line_block,jobs", CASES)
def test_variant_is_exact(spec, width, line_block, jobs):
    N = owl.best_fit(1000, spec)[1]
    exps = workloads.primes_from(9 * N, jobs)
    print("CASE", spec, width, line_block, exps[0], "x", jobs, file=sys.stderr, flush=True)
    owl.tune_set(N, width, line_block, 0)
    try:
        with owl.Batch(exps, spec) as b:
            outs, _ = b.prp(40, block_size=20, check_step=20)
        for i in {0, jobs - 1}:
            assert outs[i].res64 == oracle.gmp_res64(exps[i], 40, 40)[0], exps[i]
        assert all(o.nErrors == 0 and o.nChecks == 2 and o.maxRoe < 0.4 for o in outs)
    finally:
        owl.tune_clear()
