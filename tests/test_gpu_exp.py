"""A^h * B with its products in the fused loop, against Python integers: the smallest and largest exponents h, runs of
squarings and of products, residues 1 and M - 1, the path of a full carry per step, and a job's buffers afterwards."""
import random
import sys

import pytest

import gpuowl_amd as owl

pytestmark = pytest.mark.gpu

E = 1_000_003
M = (1 << E) - 1


def mul(x, y):
    z = x * y
    while z > M:
        z = (z & M) + (z >> E)
    return 0 if z == M else z


def power(a, h):
    r = 1
    for c in bin(h)[2:]:
        r = mul(r, r)
        if c == "1":
            r = mul(r, a)
    return r


@pytest.mark.parametrize("long_carry", [False, True])
@pytest.mark.parametrize("h", [1, 2, 3, 1 << 63, (1 << 64) - 1, 0xF0F0F0F00F0F0F0F, 0x9E3779B97F4A7C15])
def test_exp_mul(h, long_carry):
    rng = random.Random(h)
    A, B = rng.randrange(2, M), rng.randrange(2, M)
    print("CASE exp_mul", E, hex(h), long_carry, file=sys.stderr, flush=True)
    w = lambda x: owl.int_to_words(x, E)
    with owl.Gpu(E, long_carry=long_carry) as g:
        want = mul(power(A, h), B)
        assert owl.words_to_int(g.exp_mul(w(A), h, w(B))) == want
        assert g.read_int(owl.DATA) == want and g.read_int(owl.AUX) == A and g.read_int(owl.CHECK) == B
        assert owl.words_to_int(g.exp_mul(w(1), h, w(M - 1), True)) == 1
        assert owl.words_to_int(g.exp_mul(w(M - 1), h, w(B))) == (B if h % 2 == 0 else M - B)
