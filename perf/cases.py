"""The work a program has the library do, as timed cases.

A case is one call of the public API (`mm`, `mm_nt`, `bmm`, `bmm_nt`) on operands that are
already on the GPU, with the options that callers pass.  Sizes are those of the benchmark's
configurations, its sweeps, the callers under fp64-emu_amd/callers/ and the tests.

Fields of a case: `op`; `batch` (1 for the 2-D calls); `M`, `N`, `K` of one member;
`nprimes` and `corr` (0 and -1: left to the planner, as by default); `exact` (the combine);
`dist`, the operands' distribution:
  randn    iid N(0, 1)
  uniform  U(-1, 1)
  wide     sign * U[1, 2) * 2^e, e a uniform integer of [-20, 20]
  int      integers of [-2^20, 2^20], whose products the call returns exactly
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "fp64-emu_amd"))
import fp64_emu  # noqa: E402

F64 = torch.float64


def _case(name, op, batch, M, N, K, nprimes=0, corr=-1, exact=True, dist="randn"):
    case = {"op": op, "batch": batch, "M": M, "N": N, "K": K, "nprimes": nprimes, "corr": corr,
            "exact": exact, "dist": dist}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest products of the small-n table: latency and launches.
        _case("mm_64", "mm", 1, 64, 64, 64),
        # A small Gram matrix of a long operand (a CholeskyQR pass): few output tiles, deep.
        _case("mm_nt_128x128x4096", "mm_nt", 1, 128, 128, 4096),
        # A small odd-sized product with the float64 combine.
        _case("mm_nt_333x501x777", "mm_nt", 1, 333, 501, 777, exact=False),
        # Square, below the size where the chip fills (the card protocol's grid).
        _case("mm_1024", "mm", 1, 1024, 1024, 1024),
        # Walk counts by repeated squaring: integers, off the tile grid; exact results.
        _case("mm_nt_2000_int", "mm_nt", 1, 2000, 2000, 2000, dist="int"),
        # Many small members in one call (the batched sweep's smallest).
        _case("bmm_64x256", "bmm", 64, 256, 256, 256),
        # Many shallow members, each operand read in the torch.bmm layout.
        _case("bmm_nt_64x512", "bmm_nt", 64, 512, 512, 512),
        # One block column's update of the blocked Cholesky (n = 16384, t = 512, half way).
        _case("bmm_16x512x512x8192", "bmm", 16, 512, 512, 8192),
        # Square with wide exponent ranges.
        _case("mm_nt_4096_wide", "mm_nt", 1, 4096, 4096, 4096, dist="wide"),
        # The headline square product.
        _case("mm_nt_8192", "mm_nt", 1, 8192, 8192, 8192),
        # Ragged in every dimension and deep, at the reduced operating point.
        _case("mm_nt_1023x2049x32769_reduced", "mm_nt", 1, 1023, 2049, 32769, nprimes=13, corr=0,
              dist="uniform"),
        # Past the depth of one int32 accumulation (K-segmented).
        _case("mm_300x200x200000", "mm", 1, 300, 200, 200000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: small, square-ish, batched, deep or K-segmented, any size in between."""
    kind = rng.choice(["small", "square", "square", "batched", "batched", "deep", "segmented"])
    op = rng.choice(["mm", "mm_nt"])
    batch = 1
    if kind == "small":
        M, N, K = (_log_int(rng, 16, 700) for _ in range(3))
    elif kind == "square":
        n = _log_int(rng, 200, 7500)
        M, N, K = (max(16, int(n * rng.uniform(0.7, 1.3))) for _ in range(3))
        if rng.random() < 0.4:
            M, N, K = (max(256, v // 128 * 128) for v in (M, N, K))
        while M * N * K > 8192 ** 3:
            M, N, K = (int(v * 0.9) for v in (M, N, K))
    elif kind == "batched":
        op = rng.choice(["bmm", "bmm_nt"])
        n = _log_int(rng, 48, 1500)
        M, N, K = (max(16, int(n * rng.uniform(0.7, 1.3))) for _ in range(3))
        if rng.random() < 0.4:
            M, N, K = (max(64, v // 64 * 64) for v in (M, N, K))
        batch = _log_int(rng, 2, 200)
        while batch > 1 and batch * M * N * K > 4096 ** 3:
            batch //= 2
    elif kind == "deep":
        M, N = (_log_int(rng, 50, 2200) for _ in range(2))
        K = _log_int(rng, 4000, 60000)
    else:
        op = "mm"
        M, N = (_log_int(rng, 20, 500) for _ in range(2))
        K = rng.randrange(131072, 300000)
    reduced = rng.random() < 0.25
    nprimes, corr = (13, 0) if reduced else (0, -1)
    exact = rng.random() < 0.8
    dist = rng.choice(["randn", "randn", "uniform", "wide", "int"])
    if dist == "int" and (K > 4096 or reduced or not exact):
        dist = "randn"
    return _case("", op, batch, M, N, K, nprimes, corr, exact, dist)


def _shapes(case):
    b, M, N, K = case["batch"], case["M"], case["N"], case["K"]
    a, t = (M, K), ((K, N) if case["op"].endswith("_nt") else (N, K))
    return ((b, *a), (b, *t)) if case["op"].startswith("bmm") else (a, t)


def _pow2(e):
    """2^e in float64, exactly, for integer e of the normal range."""
    return (e.to(torch.int64) + 1023).bitwise_left_shift(52).view(F64)


def _operand(shape, dist, g):
    dev = g.device
    if dist == "uniform":
        return torch.rand(shape, dtype=F64, device=dev, generator=g) * 2 - 1
    if dist == "wide":
        m = 1 + torch.rand(shape, dtype=F64, device=dev, generator=g)
        e = torch.randint(-20, 21, shape, device=dev, generator=g)
        s = torch.randint(0, 2, shape, device=dev, generator=g) * 2 - 1
        return s * m * _pow2(e)
    if dist == "int":
        return torch.randint(-2 ** 20, 2 ** 20 + 1, shape, device=dev, generator=g).to(F64)
    return torch.randn(shape, dtype=F64, device=dev, generator=g)


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return tuple(_operand(s, case["dist"], g) for s in _shapes(case))


def prepare(case, seed):
    """The operands on the GPU and the call's options (only those a caller would pass)."""
    A, B = _inputs(case, seed)
    kw = {}
    if case["nprimes"]:
        kw["nprimes"] = case["nprimes"]
    if case["corr"] >= 0:
        kw["corr"] = bool(case["corr"])
    if not case["exact"]:
        kw["exact"] = False
    return {"fn": getattr(fp64_emu, case["op"]), "A": A, "B": B, "kw": kw}


def run(state):
    return state["fn"](state["A"], state["B"], **state["kw"])


def _plan(case):
    P, corr = fp64_emu.plan_config(case["K"])
    return case["nprimes"] or P, corr if case["corr"] < 0 else bool(case["corr"])


def work(case):
    """Operands read and the product written once; one int8 product per modulus and the two
    of the correction (2 operations per multiply-add)."""
    b, M, N, K = case["batch"], case["M"], case["N"], case["K"]
    P, corr = _plan(case)
    return {"bytes": 8 * b * (M * K + K * N + M * N),
            "flops": 2 * b * M * N * K * (P + (2 if corr else 0))}


def tolerance(case):
    """Integer operands give the exact product.  Otherwise the default plans are float64's
    own rounding and a little more; without the correction the operands' rounding to the
    integer width the moduli leave (about 2^-43 of the largest entry of a row) shows."""
    if case["dist"] == "int" and _plan(case)[1] and case["exact"]:
        return "exact"
    if not _plan(case)[1]:
        return {"rel": 4e-12}
    return {"rel": 1e-15}


def _slices(X, bits, count):
    """X (scaled to |x| <= 1) as `count` slices of at most `bits` bits that sum to it up to
    2^-(bits count); every slice is an integer multiple of a common power of two."""
    out, rest = [], X
    for i in range(1, count + 1):
        s = torch.round(rest * 2.0 ** (bits * i)) * 2.0 ** (-bits * i)
        out.append(s)
        rest = rest - s
    return out


def exact(case, seed):
    """The product to beyond float64: rows of A and columns of B scaled to at most 1 by powers
    of two and cut into slices whose float64 products have no rounding error, summed from the
    smallest up with the error of each sum carried."""
    A, B = _inputs(case, seed)
    Bt = B if case["op"].endswith("_nt") else B.transpose(-1, -2)

    def scale(X, dim):
        _, e = torch.frexp(X.abs().amax(dim=dim, keepdim=True))
        return e

    eA, eB = scale(A, -1), scale(Bt, -2)
    bits = (53 - math.ceil(math.log2(max(case["K"], 2)))) // 2 - 1
    count = -(-66 // bits)
    sA = _slices(A * _pow2(-eA), bits, count)
    sB = _slices(Bt * _pow2(-eB), bits, count)
    del A, Bt, B
    hi = lo = None
    for d in range(count, -1, -1):
        for i in range(count):
            if 0 <= d - i < count:
                p = torch.matmul(sA[i], sB[d - i].contiguous())
                if hi is None:
                    hi, lo = p, torch.zeros_like(p)
                    continue
                t = hi + p
                z = t - hi
                lo += (hi - (t - z)) + (p - z)
                hi = t
    return (hi + lo) * _pow2(eA) * _pow2(eB)
