"""The products this library is measured on: what a program calls it for, and what each call cannot do without.

Every case is one product C = A . B^T through the public entry point (``lib.call("hgemm_auto", ...)`` on tensors the
program keeps, or ``hgemm(A, B)``, which returns a new tensor).  The families, and where their sizes come from:

* ``square``   M = N = K, the sweep 256 ... 16384 the library is benchmarked on, up to 8192, the headline size
* ``wide``     M = N > K: an update of low rank, where writing C weighs as much as the products
* ``deep``     M = N < K: few output tiles against a long K, as in a weight gradient over many tokens
* ``prefill``  a prompt's tokens (any number of them) against a weight matrix of a feed-forward or attention layer
* ``decode``   1 ... 128 tokens of a running batch against such a matrix: B is read once and is most of the work
  (N = K = 4096 and N = 28672, K = 4096 are the benchmark's sizes; output layers have N of any parity)

``square``, ``wide`` and ``deep`` also come in sizes that no tile divides: K a multiple of 8 (rows start on 16-byte
boundaries) and odd (they do not).
"""
import math

import torch

import cuda_hgemm_amd


def _case(family, m, n, k, entry="call", name=None):
    c = {"family": family, "m": int(m), "n": int(n), "k": int(k), "entry": entry}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call of the sweep: launch latency and host work are nearly all of it
        _case("square", 256, 256, 256, name="square_256"),
        # an ordinary product of a few microseconds, as an expression of a PyTorch program
        _case("square", 1024, 1024, 1024, entry="hgemm", name="square_1024"),
        # a large product: one round of the chip
        _case("square", 4096, 4096, 4096, name="square_4096"),
        # the headline size, bound by the matrix cores
        _case("square", 8192, 8192, 8192, name="square_8192"),
        # M = N > K: 134 MB of C for 16 MB of operands
        _case("wide", 8192, 8192, 512, name="wide_8192x512"),
        # M = N < K: 64 tiles of 128 x 128 on 256 compute units
        _case("deep", 1024, 1024, 8192, name="deep_1024x8192"),
        # a prompt of 600 tokens through the up-projection of a 4096-wide feed-forward layer
        _case("prefill", 600, 14336, 4096, name="prefill_600"),
        # one token in flight against a square projection: HBM reads and latency
        _case("decode", 1, 4096, 4096, name="decode_1"),
        # a batch of 64 tokens against the same
        _case("decode", 64, 4096, 4096, name="decode_64"),
        # a batch of 16 against the benchmark's large weight matrix (235 MB)
        _case("decode", 16, 28672, 4096, name="decode_16_wide"),
        # sizes nobody rounded up: no tile divides any of the three, rows are 16-byte aligned
        _case("square", 1000, 1000, 1000, entry="hgemm", name="ragged_1000"),
        # odd sizes: rows of A, B and C start on 2-byte boundaries
        _case("square", 4095, 4095, 4095, name="odd_4095"),
    ]


_MOST_FLOPS = 2.0 * 8192 ** 3


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _rounded(rng, x, lo):
    """x as a multiple of 64 (half of the time), of 8, or odd."""
    step = rng.choice([64, 64, 8, 1])
    v = max(lo, int(x) // step * step)
    return v | 1 if step == 1 else v


def draw(rng):
    family = rng.choice(["square", "wide", "deep", "prefill", "decode", "decode"])
    entry = rng.choice(["call", "hgemm"])
    while True:
        if family == "square":
            m = n = k = _rounded(rng, _log_uniform(rng, 256, 8193), 256)
        elif family == "wide":
            m = n = _rounded(rng, _log_uniform(rng, 1024, 12289), 1024)
            k = _rounded(rng, _log_uniform(rng, 256, 1024), 256)
        elif family == "deep":
            m = n = _rounded(rng, _log_uniform(rng, 256, 1537), 256)
            k = _rounded(rng, _log_uniform(rng, 2048, 16385), 2048)
        elif family == "prefill":
            m = rng.randint(129, 4096)
            n, k = (int(_log_uniform(rng, 1024, 16385)) // 64 * 64 for _ in range(2))
        else:
            m = int(_log_uniform(rng, 1, 128.99))
            n = int(_log_uniform(rng, 1024, 65537))
            n = n | 1 if rng.random() < 0.2 else n // 64 * 64
            k = int(_log_uniform(rng, 1024, 16385)) // 64 * 64
        if 2.0 * m * n * k <= _MOST_FLOPS and n * k <= 300e6:
            return _case(family, m, n, k, entry)


def _matrix(gen, rows, cols, kind):
    """fp16, uniform in [-1, 1) as the benchmark's matrices are, or normal: activations (sigma 1), weights (0.02)."""
    x = torch.empty((rows, cols), dtype=torch.float16, device="cuda")
    if kind == "uniform":
        return x.uniform_(-1.0, 1.0, generator=gen)
    return x.normal_(0.0, 1.0 if kind == "activations" else 0.02, generator=gen)


def prepare(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    layer = case["family"] in ("prefill", "decode")
    state = {"lib": cuda_hgemm_amd.library(), "m": m, "n": n, "k": k, "entry": case["entry"],
             "A": _matrix(gen, m, k, "activations" if layer else "uniform"),
             "B": _matrix(gen, n, k, "weights" if layer else "uniform")}
    if case["entry"] == "call":
        state["C"] = torch.empty((m, n), dtype=torch.float16, device="cuda")
    return state


def run(state):
    if state["entry"] == "hgemm":
        return cuda_hgemm_amd.hgemm(state["A"], state["B"])
    state["lib"].call("hgemm_auto", state["A"], state["B"], state["C"], state["m"], state["n"], state["k"])
    return state["C"]


def work(case):
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2 * m * n * k}


def tolerance(case):
    # fp32 sums rounded once to fp16: against the same product in 64 bits every size shows 2.1e-4 (the rounding to 11
    # bits); the largest single difference is half a unit in the last place of the largest output
    return {"rel": 8e-4, "max": 8e-3}
