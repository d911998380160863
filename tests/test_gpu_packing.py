"""Residue words <-> balanced digits on the device, against the oracle: words of every pattern whose carries or borrows
run far (a long run of digits that pass them on is the host's to decide), digits that no normalized state holds, and
shapes and exponents from 3 to 19 bits per word."""
import random
import sys

import pytest

import gpuowl_amd as owl
import oracle
from gpuowl_amd import workloads

pytestmark = pytest.mark.gpu


def patterns(E, N, rng):
    full = (1 << E) - 1
    lo, pos = E // N, lambda k: -(-k * E // N)
    halves = sum(((1 << (pos(k + 1) - pos(k) - 1)) - 1) << pos(k) for k in range(N // 2, N // 2 + 40))
    few = sum(((1 << (pos(k + 1) - pos(k) - 1)) - 1) << pos(k) for k in range(100, 108))
    return [rng.getrandbits(E) % full, 1, 3, full - 1, 1 << (E - 1), (1 << (E - 1)) - 1, rng.getrandbits(40), halves,
            halves | 1 << pos(N // 2), rng.getrandbits(E) >> lo << lo & ~(full >> 100 << 50), few | 1 << (pos(100) - 1),
            full ^ (1 << (E // 2))]


@pytest.mark.parametrize("spec,bits", [("256:2:256", 3.3), ("256:2:256", 18.1), ("256:9:256", 12.7), ("512:5:256", 17.03)])
def test_words_and_digits(spec, bits):
    N = owl.best_fit(1000, spec)[1]
    E = workloads.primes_from(int(bits * N), 1)[0]
    rng = random.Random(E)
    print("CASE", spec, E, file=sys.stderr, flush=True)
    with owl.Gpu(E, spec) as g:
        n = owl.n_words(E)
        for i, x in enumerate(patterns(E, N, rng)):
            words = owl.int_to_words(x, E)
            g.write_words(owl.DATA, words)
            assert g.read_digits() == list(oracle.expand(words, N, E)), i
            assert g.read_words() == words, i
        g.write_words(owl.DATA, [0] * n)
        assert g.read_words() == [0] * n and not any(g.read_digits())
        # bits above E come back in digit 0
        words = owl.int_to_words(rng.getrandbits(E), E)
        words[-1] |= 3 << E % 32 if E % 32 < 30 else 0
        g.write_words(owl.DATA, words)
        assert g.read_digits() == list(oracle.expand(words, N, E))
        with pytest.raises(owl.OwlError, match="too many words"):
            g.write_words(owl.DATA, words + [0])
        with pytest.raises(owl.OwlError, match="too few words"):
            g.write_words(owl.DATA, words[:-1])


def test_digits_the_host_decides():
    spec = "256:2:256"
    N = owl.best_fit(1000, spec)[1]
    E = workloads.primes_from(9 * N + 5, 1)[0]
    rng = random.Random(7)
    d = oracle.expand(owl.int_to_words(rng.getrandbits(E), E), N, E)
    with owl.Gpu(E, spec) as g:
        for lead, sign in ((5, 1), (5, -1), (40, 1), (40, -1)):  # low zeros, a borrow from the top or none
            t = [0] * lead + list(d[lead:])
            t[-1] = sign * max(abs(t[-1]), 1)
            g.write_digits(owl.DATA, t)
            assert g.read_words() == list(oracle.compact(t, N, E)), (lead, sign)
        t = list(d)
        t[1000] = (1 << 9) - 1  # not balanced, but a digit
        g.write_digits(owl.DATA, t)
        assert g.read_words() == list(oracle.compact(t, N, E))
        t[1000] = 1 << 20
        g.write_digits(owl.DATA, t)
        with pytest.raises(owl.OwlError, match="digit out of range"):
            g.read_words()
