"""Every compiled variant of the squaring's passes (complex or split exchanges, plain or non-temporal accesses) against GMP, by
the name of the kernel that a launch runs: for every height of the column pass and every 16-element row pass, the
smallest number of jobs for which the engine picks each variant, run as a batch of that many jobs. The split exchanges of
short columns are not compiled; the complex ones of tall columns with plain accesses run under OWL_COL_ONE_PAIR only."""
import functools
import re
import sys

import pytest

import gpuowl_amd as owl
import oracle
from gpuowl_amd import workloads

pytestmark = pytest.mark.gpu

COLUMNS, ROWS = {}, {}
for n in owl.kernel_names():
    if m := re.fullmatch(r"col(?:cp|cn|sn)(\d+)|colx(\d+)m", n):
        COLUMNS.setdefault(int(m.group(1) or m.group(2)), set()).add(n)
    elif m := re.fullmatch(r"row(?:cp|cn|sp|sn)(\d+)r(\d+)", n):
        ROWS.setdefault((int(m.group(1)), int(m.group(2))), set()).add(n)
ONE_PAIR, MOST = 8, 64


def reference_spec(nd):
    """A reference FFT spec (width:middle:height) with width*middle*height == nd."""
    fmt = {256: "256", 512: "512", 1024: "1K", 4096: "4K"}
    return next((f"{fmt[a]}:{nd // (a * c)}:{fmt[c]}" for a in (256, 512, 1024, 4096) for c in (256, 512, 1024)
                 if nd % (a * c) == 0 and 1 <= nd // (a * c) <= 16), None)


@functools.lru_cache(maxsize=None)
def gmp(E, iters):
    return oracle.gmp_res64(E, iters, iters)[0]


def check_all(names, geometries, which):
    """Runs every one of `names`: geometries (spec, W, R, flags) in turn, job counts from 1 up."""
    left = set(names)
    for spec, W, R, flags in geometries:
        N = owl.best_fit(1000, spec)[1]
        exps = workloads.primes_from(5 * N, MOST)
        owl.tune_set(N, W, R, flags)
        try:
            with owl.Gpu(exps[0], spec) as g:
                assert (g.W, g.R, g.long_carry) == (W, R, False)
                jobs = {}
                for n in range(1, MOST + 1):
                    jobs.setdefault(g.launched(n)[which], n)
            for name in sorted(left & set(jobs)):
                n = jobs[name]
                print("CASE", name, spec, W, R, flags, exps[0], "x", n, file=sys.stderr, flush=True)
                with owl.Batch(exps[:n], spec) as b:
                    assert b.launched(0)[which] == name
                    outs, _ = b.prp(28, block_size=14, check_step=14)
                assert outs[0].res64 == gmp(exps[0], 28)
                assert all(o.nErrors == 0 and o.nChecks == 2 and o.maxRoe < 0.4 for o in outs)
                left.discard(name)
        finally:
            owl.tune_clear()
        if not left:
            return
    assert not left, f"no launch runs {left}"


@pytest.mark.parametrize("H", sorted(COLUMNS))
def test_every_column_variant_is_exact(H):
    W = next(w for w in (256, 1024, 512) if reference_spec(w * H))
    R = 8 if W == 256 and H % 128 == 0 else 2
    check_all(COLUMNS[H], [(reference_spec(W * H), W, R, flags) for flags in (0, ONE_PAIR)], 1)


@pytest.mark.parametrize("W,R", sorted(ROWS))
def test_every_row_variant_is_exact(W, R):
    check_all(ROWS[W, R], [(reference_spec(W * H), W, R, 0) for H in (512, 1024, 256)], 0)
