"""Performance cases of the modular-squaring engine: what programs that use it have it do.

A case names one call pattern ("kind"), an exponent (or a list of them) and a count of squarings.
Residues are random E-bit values, as they are from a test's first few dozen iterations on. Every
pass ends with the residue on the host as 32-bit words, which is what a program saves, compares
or hashes; batches and the server return what their interfaces return, the final res64 values.

The ranges: exponents from 1,000,000 to 140,000,000 (FFTs of 256K to 7.5M words, the sizes that the
engine's exponent selection, its tests and its benchmark cover), low bits per word at the bottom of
the range where 256K words is the smallest FFT, every FFT length in between.
"""
import ctypes as C
import math
import random

import numpy as np

import gpuowl_amd as owl
from gpuowl_amd import workloads
from gpuowl_amd._lib import check

LO, HI = 1_000_000, 140_000_000
U32P = C.POINTER(C.c_uint32)


def _prime(n):
    return workloads.next_prime(int(n))


def listed():
    return [
        # One product of two residues at the benchmark's small exponent: the smallest call, a Gerbicz
        # update or one proof multiply, whose launches and latency are not hidden by anything.
        {"name": "mul_4m", "kind": "mul", "E": _prime(4_000_000)},
        # Lucas-Lehmer squarings at the smallest FFT with few bits per word.
        {"name": "ll_2m", "kind": "loop", "E": _prime(2_000_000), "iters": 1000, "ll": True},
        # The benchmark's small PRP exponent: 256K words, steady squarings.
        {"name": "prp_4m", "kind": "loop", "E": _prime(4_000_000), "iters": 2000, "ll": False},
        # A 512K-word test, the middle of the small exponents.
        {"name": "prp_9m", "kind": "loop", "E": _prime(9_000_000), "iters": 1000, "ll": False},
        # The batch benchmark's exponent run alone: 1.5M words.
        {"name": "prp_20m", "kind": "loop", "E": _prime(20_000_000), "iters": 1000, "ll": False},
        # Double-check size, Lucas-Lehmer, a tall FFT shape.
        {"name": "ll_57m", "kind": "loop", "E": _prime(57_000_000), "iters": 1000, "ll": True},
        # The headline: a first-time PRP test at 7.5M words, one block of squarings.
        {"name": "prp_139m", "kind": "loop", "E": _prime(139_000_000), "iters": 1000, "ll": False},
        # A whole PRP call with Gerbicz updates every block and a verification at the end.
        {"name": "prp_checked_40m", "kind": "prp", "E": _prime(40_000_000), "iters": 1000, "block": 200},
        # One step of proof making or verification: A^h * B for a 64-bit h.
        {"name": "proof_step_9m", "kind": "exp", "E": _prime(9_500_000)},
        # A checkpoint at the headline size restored to the GPU and read back.
        {"name": "checkpoint_139m", "kind": "state", "E": _prime(139_000_000)},
        # 64 exponents advanced together, the uniform batch of the benchmark.
        {"name": "batch_64x20m", "kind": "batch", "E": _prime(20_000_000), "span": 1.0, "jobs": 64, "iters": 500},
        # The serving loop: requests of uneven exponents and both kinds share a round of 1,000.
        {"name": "serve_uneven", "kind": "serve", "E": _prime(2_000_000), "span": 30.0, "jobs": 12, "iters": 1000},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["loop"] * 5 + ["prp", "mul", "exp", "state", "batch", "serve"])
    E = _prime(_log_uniform(rng, LO, HI * 0.99))
    # squarings of one pass: fewer for larger exponents, so that a pass stays near a tenth of a second
    iters = int(min(2000, max(100, 1.2e11 / E * rng.uniform(0.5, 1.0))))
    if kind == "loop":
        return {"kind": kind, "E": E, "iters": iters, "ll": rng.random() < 0.5}
    if kind == "prp":
        block = max(20, iters // 8)
        return {"kind": kind, "E": E, "iters": 4 * block, "block": block}
    if kind in ("mul", "state"):
        return {"kind": kind, "E": E}
    if kind == "exp":
        return {"kind": kind, "E": _prime(_log_uniform(rng, LO, 60e6))}
    # uneven groups: exponents log-uniform over a factor of span
    span = rng.choice([1.0, 4.0, 20.0])
    jobs = rng.randrange(4, 25)
    E = _prime(_log_uniform(rng, LO, 50e6 / span))
    return {"kind": kind, "E": E, "span": span, "jobs": jobs, "iters": rng.randrange(150, 400)}


def _exponents(case, seed):
    """The exponents of one set of inputs: primes just above the case's (or, for the groups of
    jobs, log-uniform over its span), other ones for another seed."""
    rng = random.Random(seed)
    if case["kind"] == "prp":
        return [_prime(case["E"] + 2 * rng.randrange(1000))]
    out = []
    while len(out) < case["jobs"]:
        if case["span"] == 1.0:
            p = _prime(out[-1] + 1 if out else case["E"] + 2 * rng.randrange(1000))
        else:
            p = _prime(_log_uniform(rng, case["E"], case["E"] * case["span"]))
        if p not in out:
            out.append(p)
    return out


def _residues(case, seed, n):
    """n random residues below 2^E as little-endian 32-bit words."""
    E = case["E"]
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        w = rng.integers(0, 1 << 32, owl.n_words(E), dtype=np.uint32)
        w[-1] &= np.uint32((1 << (E % 32)) - 1)
        out.append(w)
    return out


def _write(g, buf, words):
    check(g.lib.owl_gpu_write_words(g.h, buf, words.ctypes.data_as(U32P), len(words)))


def _read(g, buf, room=0):
    """The residue in buf as n_words(E) words, followed by zeros up to `room` words."""
    n = owl.n_words(g.E)
    out = np.zeros(max(n, room), dtype=np.uint32)
    zero = C.c_int()
    check(g.lib.owl_gpu_read_words(g.h, buf, out.ctypes.data_as(U32P), n, C.byref(zero)))
    if zero.value:
        out[:] = 0
    return out


def _res64(values):
    """64-bit residues as pairs of 32-bit words."""
    return np.array(values, dtype=np.uint64).view(np.uint32)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "batch":
        s["batch"] = owl.Batch(_exponents(case, seed))
    elif kind == "serve":
        s["server"] = owl.Server(block_size=case["iters"])
        s["exponents"] = _exponents(case, seed)
    elif kind == "prp":
        s["gpu"] = owl.Gpu(_exponents(case, seed)[0])
    else:
        s["gpu"] = owl.Gpu(case["E"])
        s["x"] = _residues(case, seed, 1 if kind in ("loop", "state") else 2)
        if kind in ("loop", "mul"):
            _write(s["gpu"], owl.DATA, s["x"][0])
        if kind == "mul":
            _write(s["gpu"], owl.CHECK, s["x"][1])
        if kind == "exp":
            s["h"] = random.Random(seed).getrandbits(63) | 1 << 63
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "loop":
        g = state["gpu"]
        g.square_loop(owl.AUX, owl.DATA, 0, case["iters"], ll=case["ll"])
        return _read(g, owl.AUX)
    if kind == "mul":
        g = state["gpu"]
        g.copy(owl.AUX, owl.CHECK)
        g.mod_mul(owl.AUX, owl.DATA)
        return _read(g, owl.AUX)
    if kind == "prp":
        g = state["gpu"]
        out, _ = g.prp(case["iters"], block_size=case["block"], check_step=case["iters"])
        return {"k": out.k, "res64": _res64([out.res64]), "checks": out.nChecks, "errors": out.nErrors,
                "x": _read(g, owl.DATA, owl.n_words(case["E"] + 8192))}
    if kind == "exp":
        g, (a, b) = state["gpu"], state["x"]
        out = np.empty(len(a), dtype=np.uint32)
        check(g.lib.owl_gpu_exp_mul(g.h, a.ctypes.data_as(U32P), state["h"], b.ctypes.data_as(U32P), 0,
                                    out.ctypes.data_as(U32P), len(out)))
        return out
    if kind == "state":
        g = state["gpu"]
        _write(g, owl.DATA, state["x"][0])
        return _read(g, owl.DATA)
    if kind == "batch":
        outs, _ = state["batch"].ll(case["iters"])
        return _res64([o.res64 for o in outs])
    srv = state["server"]
    order = {}
    for i, E in enumerate(state["exponents"]):
        order[srv.submit(E, "ll" if i % 2 else "prp", case["iters"])] = i
    done = {order[r["id"]]: r for r in srv.drain()}
    return {"res64": _res64([done[i]["res64"] for i in sorted(done)]), "errors": [done[i]["nErrors"] for i in sorted(done)]}


def _squaring(E):
    """Bytes and FP64 operations of one squaring mod 2^E - 1. The transform is longer than what one
    workgroup can hold, so its words (8 bytes each) cross memory in two passes, each read once and
    written once; two complex FFTs of N/2 points (5 n log2 n each) and about 25 operations per
    word for weights, carries and the pointwise square."""
    N = owl.best_fit(E)[1]
    return 32 * N, 5 * N * math.log2(N / 2) + 25 * N


def work(case):
    kind, E = case["kind"], case["E"]
    host = 4 * owl.n_words(E)  # one residue in 32-bit words
    b, f = _squaring(E)
    if kind == "loop":
        return {"bytes": case["iters"] * b + host, "flops": case["iters"] * f}
    if kind == "mul":
        return {"bytes": 2 * b + 3 * host, "flops": 1.5 * f}
    if kind == "prp":  # the squarings, the same count again over check's block, a product per block
        n = case["iters"] + case["block"] + 2 * (case["iters"] // case["block"] + 1)
        return {"bytes": n * b + host, "flops": n * f}
    if kind == "exp":  # 63 squarings, about half as many products, one more product
        return {"bytes": (63 + 2 * 33) * b + 3 * host, "flops": (63 + 1.5 * 33) * f}
    if kind == "state":  # words to digits and back, the digits written and read once
        N = owl.best_fit(E)[1]
        return {"bytes": 2 * host + 2 * 4 * N, "flops": 4 * N}
    total_b = total_f = 0
    for E in _exponents(case, 0):
        b, f = _squaring(E)
        # every second served request is a PRP test whose block is squared again to check it
        n = case["iters"] * (1 if kind == "batch" else 1.5)
        total_b, total_f = total_b + n * b, total_f + n * f
    return {"bytes": total_b, "flops": total_f}


def _to_int(w):
    return int.from_bytes(w.tobytes(), "little")


def exact(case, seed):
    """A product by Python's integers, a checkpoint read back as it was written; a run of squarings
    has no value that plain code reaches in seconds."""
    E = case["E"]
    if case["kind"] == "state":
        return _residues(case, seed, 1)[0]
    if case["kind"] == "mul" and E < 30_000_000:
        a, b = (_to_int(w) for w in _residues(case, seed, 2))
        x = a * b
        m = (1 << E) - 1
        while x > m:
            x = (x & m) + (x >> E)
        x = 0 if x == m else x
        return np.frombuffer(x.to_bytes(4 * owl.n_words(E), "little"), dtype=np.uint32).copy()
    return None
