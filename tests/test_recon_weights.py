"""CPU tier: the remainder-weight combine of the reconstruction (crt_values and
crt_combine in remainder_weights.h) against exact integers: three 39-bit slices
of the weights, any residue representatives (a K-split's sums among them), the
correction, and a single rounding -- at range ends, ties and cancellations.
The kernels' own code, compiled for the host, and its operations restated in
correctly rounded float64 (with the slices' bounds).  Tolerance: none (the same
bits)."""
import ctypes
import math
import os
import random
import subprocess
from fractions import Fraction

import pytest

import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "fp64-emu_amd", "csrc")
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
BITS = 39


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def _slices(v):
    out = []
    for _ in range(2):
        low = (v + (1 << (BITS - 1))) % (1 << BITS) - (1 << (BITS - 1))
        out.insert(0, float(low))
        v = (v - low) >> BITS
    return [float(v)] + out


def _weights(primes):
    M = math.prod(primes)
    W = [M // p * pow(M // p, -1, p) for p in primes]
    W = [w - M if 2 * w > M else w for w in W]
    return M, W


def _combine(s, cv, cshift, M):
    """crt_combine before its final scaling."""
    kB, magic = 2.0 ** BITS, 6755399441055744.0
    m = _slices(M)
    s1, s2, s3 = s
    q = _fma(_fma(s1, kB, s2), 2.0 ** BITS / float(M), magic) - magic
    s1, s2, s3 = (_fma(-q, mi, si) for mi, si in zip(m, (s1, s2, s3)))
    h = _fma(s1, kB, s2)
    l = s2 - _fma(s1, -kB, h)
    d = math.ldexp(float(cv), cshift)
    u = d + s3
    v = s3 - (u - d)
    p = _fma(l, kB, u)
    e = u - _fma(l, -kB, p)
    h2 = _fma(h, kB, p)
    p2 = p - _fma(h, -kB, h2)
    t = e + v
    y = p2 + t
    err = t - (y - p2)
    if err != 0.0 and int(math.frexp(y)[0] * 2 ** 53) % 2 == 0:   # to odd
        away = (err > 0.0) == (y > 0.0)
        y = math.copysign(math.nextafter(abs(y), math.inf if away else 0.0), y)
    return h2 + y


FOLDS = [(12, 1), (13, 1), (14, 1), (15, 1), (13, 16), (14, 16), (15, 8)]


def _cases(P, fold):
    """(X, cv, cshift, residues): X = sum of the residues at their weights, mod M."""
    primes = [int(p) for p in O.PRIMES[:P]]
    M, _ = _weights(primes)
    rng = random.Random(100 * P + fold)
    lim = 36 * M // 100
    for it in range(600):
        cs, cv = rng.randint(1, 38), rng.randint(-2 ** 32, 2 ** 32) >> rng.randint(0, 32)
        X = rng.randint(-lim, lim) >> rng.choice([0, 0, 1, 30, 60, 100])
        if it % 5 == 1:      # cancels against the correction
            X = -(cv << cs) + rng.randint(-2 ** 20, 2 ** 20)
        elif it % 5 == 2:    # near a tie of the result
            k = rng.randint(1, 55)
            X = (rng.randint(-2 ** 53, 2 ** 53) << k) + (1 << (k - 1)) + rng.randint(-1, 1) - (cv << cs)
        elif it % 5 == 3:
            X = rng.choice([0, 1, -1, lim, -lim])
        if abs(X) > lim:
            continue
        r = []
        for p in primes:     # a sum of `fold` representatives in [-p/2, p/2]
            parts = [rng.choice([-(p // 2), (p - 1) // 2, rng.randint(-(p // 2), (p - 1) // 2)])
                     for _ in range(fold - 1)]
            last = (X - sum(parts)) % p
            r.append(sum(parts) + (last - p if last > (p - 1) // 2 else last))
        yield X, cv, cs, r


def _same(a, b):
    return a == b and math.copysign(1.0, a) == math.copysign(1.0, b)


@pytest.mark.parametrize("P,fold", FOLDS)
def test_weight_combine_rounds_once(P, fold):
    primes = [int(p) for p in O.PRIMES[:P]]
    M, W = _weights(primes)
    slices = [_slices(w) for w in W]
    for i in range(3):   # every partial sum, before and after q M, is an exact float64
        bound = fold * sum(p // 2 * abs(s[i]) for p, s in zip(primes, slices))
        q = fold * sum(p // 2 * abs(w) for p, w in zip(primes, W)) // M + 1
        assert bound + q * abs(_slices(M)[i]) < 2 ** 53
    for X, cv, cs, r in _cases(P, fold):
        s = [float(sum(Fraction(ri) * Fraction(si[i]) for ri, si in zip(r, slices))) for i in range(3)]
        assert _same(_combine(s, cv, cs, M), float(Fraction(X + (cv << cs)))), (X, cv, cs)


HOST = """
#include "remainder_weights.h"
template <int kP> static double value(const int* r, double cv, int cshift, int sh) {
  const double cvs[1] = {cv};
  const int shs[1] = {sh};
  double out[1];
  crt_values<kP, 1>([&](int t, int) { return r[t]; }, cvs, cshift, shs, out);
  return out[0];
}
extern "C" double host_value(int P, const int* r, double cv, int cshift, int sh) {
  switch (P) {
    case 12: return value<12>(r, cv, cshift, sh);
    case 13: return value<13>(r, cv, cshift, sh);
    case 14: return value<14>(r, cv, cshift, sh);
    default: return value<15>(r, cv, cshift, sh);
  }
}
extern "C" int host_exact(int P, int fold) { return crt_exact(P, fold); }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("weights")
    (d / "host.hip").write_text(HOST)
    subprocess.run([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-ffp-contract=off", "-shared",
                    f"-I{CSRC}", f"-I{ROOT}/include", str(d / "host.hip"), "-o", str(d / "host.so")], check=True)
    L = ctypes.CDLL(str(d / "host.so"))
    L.host_value.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_double, ctypes.c_int, ctypes.c_int]
    L.host_value.restype = ctypes.c_double
    return L


@pytest.mark.parametrize("P,fold", FOLDS)
def test_compiled_combine_rounds_once(host, P, fold):
    assert host.host_exact(P, fold)
    for i, (X, cv, cs, r) in enumerate(_cases(P, fold)):
        sh = (0, -7, -60, 40)[i % 4]
        got = host.host_value(P, (ctypes.c_int * P)(*r), float(cv), cs, sh)
        assert _same(got, math.ldexp(float(Fraction(X + (cv << cs))), sh)), (X, cv, cs, sh)


def test_compiled_combine_bounds(host):
    """Exact for sums of residues to sixteen splits at 12 to 14 moduli, to eight at 15; no
    other modulus count."""
    exact = {(P, f) for P in range(1, 21) for f in (1, 2, 4, 8, 16) if host.host_exact(P, f)}
    want = {(P, f) for P in (12, 13, 14) for f in (1, 2, 4, 8, 16)} | {(15, f) for f in (1, 2, 4, 8)}
    assert exact == want
