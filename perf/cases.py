"""Timed cases of the squaring engine: what its users run, over the whole range of lengths.

A user's program holds one test per exponent (`LucasPRP`), advances it many squarings at a
time and reads the whole residue back at a checkpoint; or holds many tests in a `Batch`; or
runs a PRP test under the Gerbicz check; or squares a residue in its own device memory
(`lnt_iterate_static`).  A pass is one such stretch: k squarings, then the residue as
canonical digits (or, for the static entry point, the caller's buffer).  The exponents and
lengths are those of the tests, the bench and the workloads of this repository.
"""
import ctypes
import math

import numpy as np
import torch

import cuda_amd

# What the cases stand for:
#   ll512, prp1024, ll4096   tests of small exponents that run in one workgroup, where the
#                            latency of one squaring counts (the small Mersenne fixtures,
#                            the full test of M86243)
#   static2p13               a residue in the caller's memory, short calls on one stream
#   ll2p16, prp2p18, ll2p20  the lengths of the batched workload, one test at a time
#   ll2p22                   the headline throughput configuration
#   checked2p23              a PRP chunk with Gerbicz block products and one check
#   prp2p25                  a residue far beyond the caches
#   batch_served             the LL requests of the served mix in one batch (2^11 .. 2^14)
#   batch_mixed              the batched workload's spread of lengths (2^16 .. 2^20)
_LISTED = [
    {"name": "ll512", "kind": "single", "p": 9689, "log_n": 9, "prp": False, "k": 256},
    {"name": "prp1024", "kind": "single", "p": 19937, "log_n": 10, "prp": True, "k": 256},
    {"name": "ll4096", "kind": "single", "p": 86243, "log_n": 12, "prp": False, "k": 512},
    {"name": "static2p13", "kind": "static", "p": 132049, "log_n": 13, "prp": True, "k": 100},
    {"name": "ll2p16", "kind": "single", "p": 1000003, "log_n": 16, "prp": False, "k": 1000},
    {"name": "prp2p18", "kind": "single", "p": 4000037, "log_n": 18, "prp": True, "k": 1000},
    {"name": "ll2p20", "kind": "single", "p": 16000057, "log_n": 20, "prp": False, "k": 2000},
    {"name": "ll2p22", "kind": "single", "p": 70000027, "log_n": 22, "prp": False, "k": 2000},
    {"name": "checked2p23", "kind": "checked", "p": 140000041, "log_n": 23, "prp": True, "k": 1000, "block": 500},
    {"name": "prp2p25", "kind": "single", "p": 637534199, "log_n": 25, "prp": True, "k": 300},
    {"name": "batch_served", "kind": "batch", "p": 50021, "p_hi": 250007, "tests": 24, "prp": False, "k": 500},
    {"name": "batch_mixed", "kind": "batch", "p": 1000003, "p_hi": 18000041, "tests": 12, "prp": False, "k": 300},
]


def listed():
    return [dict(c) for c in _LISTED]


def _log_length(p):
    """log2 of the length the engine picks for exponent p: the smallest L with p <= 32 * 2^L
    whose digits w = ceil(p / 2^L) satisfy (2^w - 1)^2 < P / 2^(L + 1), one more otherwise."""
    L = 0
    while (32 << L) < p:
        L += 1
    w = -(-p >> L)
    if ((1 << w) - 1) ** 2 << (L + 1) >= (1 << 64) - (1 << 32) + 1:
        L += 1
    return L


def draw(rng):
    """Another case of the same ranges: exponents log-uniform (any odd number, prime or not),
    at the default length or twice it (fewer bits per digit), LL or PRP."""
    def exponent(lo, hi):
        return int(lo * math.exp(math.log(hi / lo) * rng.random())) | 1
    kind = rng.choice(["single", "single", "single", "single", "static", "static", "batch", "checked"])
    prp = rng.random() < 0.5 or kind == "checked"
    if kind == "batch":
        lo = exponent(3000, 4000000)
        hi = int(lo * (2 + 6 * rng.random())) | 1
        tests = rng.randint(3, 24)
        k = max(30, min(600, int(2 ** 31 / (tests << _log_length(hi)))))
        return {"kind": kind, "p": lo, "p_hi": hi, "tests": tests, "prp": prp, "k": k}
    p = exponent(600, {"static": 15000000, "checked": 80000000, "single": 90000000}[kind])
    log_n = _log_length(p)
    if rng.random() < 0.25 and log_n < (20 if kind == "static" else 22):
        log_n += 1  # a longer transform than the exponent needs
    k = max(20, min(rng.randint(200, 1500), 2 ** 32 >> log_n))
    case = {"kind": kind, "p": p, "log_n": log_n, "prp": prp, "k": k}
    if kind == "checked":
        case["block"] = max(10, k // 2)
        case["k"] = 2 * case["block"]
    return case


def _widths(p, n):
    i = np.arange(n + 1, dtype=np.int64)
    e = (p * i + n - 1) // n
    return np.diff(e)


def _digits(p, n, seed):
    """A residue as it is in the middle of a test: every digit uniform over its width."""
    w = _widths(p, n)
    rng = np.random.default_rng([int(seed) & 0xFFFFFFFF, p, n])
    d = rng.integers(0, 1 << int(w.max()), n, dtype=np.int64)
    return (d & ((np.int64(1) << w) - 1)).astype(np.uint64)


def _exponents(case):
    """The batch's exponents: spread evenly over the logarithm of [p, p_hi]."""
    lo, hi, m = case["p"], case["p_hi"], case["tests"]
    return [int(lo * math.exp(math.log(hi / lo) * (i + 0.5) / m)) | 1 for i in range(m)]


def prepare(case, seed):
    if case["kind"] == "batch":
        ps = _exponents(case)
        tests = [cuda_amd.LucasPRP(p, prp=case["prp"]) for p in ps]
        batch = cuda_amd.Batch()
        for i, t in enumerate(tests):
            t.set_digits(_digits(t.p, t.n, seed + 1000 * i))
            batch.add(t)
        return {"case": case, "tests": tests, "batch": batch}
    p, n = case["p"], 1 << case["log_n"]
    d = _digits(p, n, seed)
    if case["kind"] == "static":
        lib = cuda_amd.load()
        lib.lnt_iterate_static.argtypes = [ctypes.c_uint32, ctypes.c_int, ctypes.c_void_p, ctypes.c_size_t,
                                           ctypes.c_uint32, ctypes.c_void_p]
        return {"case": case, "lib": lib, "x": torch.from_numpy(d.astype(np.int64)).cuda()}
    t = cuda_amd.LucasPRP(p, n, prp=case["prp"])
    t.set_digits(d)
    if case["kind"] == "checked":
        t.gerbicz_begin(case["block"], 2)
    return {"case": case, "test": t}


def _read(t):
    return np.frombuffer(t.get_digits_buffer(), dtype=np.int64)


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        state["batch"].iterate(case["k"])
        return [_read(t) for t in state["tests"]]
    if case["kind"] == "static":
        x = state["x"]
        rc = state["lib"].lnt_iterate_static(case["p"], int(case["prp"]), x.data_ptr(), x.numel(), case["k"],
                                             torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError("lnt_iterate_static: %d" % rc)
        return x
    t = state["test"]
    if case["kind"] == "checked":
        t.gerbicz_iterate(case["k"])
        st = t.gerbicz_stats()
        product = st["checkpoint_res64"]  # low 64 bits of the verified block product
        return {"digits": _read(t), "product": product - (1 << 64) if product >> 63 else product,
                "rollbacks": st["rollbacks"]}
    t.iterate(case["k"])
    return _read(t)


def work(case):
    """Bytes: a residue that fits one compute unit is read and written once per pass; a larger
    one is read and written once per squaring.  Operations: the modular multiplications and
    additions of two transforms (n/2 log2 n butterflies each), the square and the weights."""
    if case["kind"] == "batch":
        shapes = [(1 << _log_length(p), case["k"]) for p in _exponents(case)]
    else:
        k = case["k"]
        if case["kind"] == "checked":  # the squarings of the check, and two products per block
            k += case["block"] + 4
        shapes = [(1 << case["log_n"], k)]
    return {"bytes": sum(16 * n * (k if n > 4096 else 1) for n, k in shapes),
            "flops": sum(k * n * (3 * int(math.log2(n)) + 3) for n, k in shapes)}


def tolerance(case):
    return "exact"  # residues of integer arithmetic


def exact(case, seed):
    """The residue by Python's integers, for exponents where that takes a few seconds."""
    if case["kind"] != "single" or case["k"] * float(case["p"]) ** 1.585 > 2e11:
        return None
    p, n = case["p"], 1 << case["log_n"]
    e = [-(-p * i // n) for i in range(n + 1)]
    mask = (1 << p) - 1
    v = 0
    for i, d in enumerate(_digits(p, n, seed).tolist()):
        v |= d << e[i]
    for _ in range(case["k"]):
        v = v * v
        v = (v & mask) + (v >> p)
        v = (v & mask) + (v >> p)
        if not case["prp"]:
            v = v - 2 if v >= 2 else v - 2 + mask
    if v == mask:
        v = 0
    return np.array([(v >> e[i]) & ((1 << (e[i + 1] - e[i])) - 1) for i in range(n)], dtype=np.int64)
