"""GPU tier: fp64emu_product, the form the torch ops call, against the staged
entry points bit for bit, on a workspace filled with a nonzero byte (rows of
the planes past the operands are never written there)."""
import pytest
import torch

import oracle as O
from fp64_emu import capi
from parity_util import bits_equal

pytestmark = pytest.mark.gpu


def _pair(kind, batch, M, N, K, seed, dev):
    g = torch.Generator().manual_seed(seed)
    lead = (batch,) if kind.startswith("bmm") else ()
    A = torch.randn(lead + (M, K), dtype=torch.float64, generator=g)
    B = torch.randn(lead + ((K, N) if kind.endswith("_nt") else (N, K)), dtype=torch.float64, generator=g)
    return A.to(dev), B.to(dev)


def _check(dev, kind, batch, M, N, K, P, corr, exact=True):
    print(f"case product {kind} b={batch} {M}x{N}x{K} P={P} corr={corr} exact={exact}", flush=True)
    A, B = _pair(kind, batch, M, N, K, M + 3 * N + K, dev)
    primes = O.PRIMES[:P]
    got = capi.product(kind, A, B, primes, exact=exact, use_corr=corr, fill=0x5A)
    ref, _, _ = capi.run(kind, A, B, primes, exact=exact, use_corr=corr)
    torch.cuda.synchronize()
    assert bits_equal(got.cpu().numpy(), ref.cpu().numpy())
    return A, B, got


# Past one launch's depth: whole-K splits (128 x 128 and 256 x 256 tiles, a last
# split shorter than the others, more than eight splits at 15 moduli, a mixed last
# column), against the segmented form.
@pytest.mark.parametrize("kind,batch,M,N,K,P,corr,exact", [
    ("mm", 1, 40, 24, 140_000, 15, True, True),
    ("mm", 1, 129, 300, 131_072, 16, True, True),
    ("mm", 1, 250, 500, 131_137, 13, False, True),
    ("mm", 1, 256, 300, 150_000, 15, True, False),
    ("bmm", 2, 24, 16, 135_000, 15, True, True),
    ("mm", 1, 3, 2, 1_200_000, 15, True, True),
    ("mm", 1, 2, 3, 2_096_200, 15, True, True),     # past the whole-K bound: segmented
])
def test_whole_k(dev, kind, batch, M, N, K, P, corr, exact):
    _check(dev, kind, batch, M, N, K, P, corr, exact)


# Rows that end inside 64-row groups, 128-row tiles and 256-row tiles.
@pytest.mark.parametrize("kind,batch,M,N,K,P,corr", [
    ("mm_nt", 1, 1, 1, 1, 14, True),
    ("mm", 1, 65, 129, 63, 14, True),
    ("mm_nt", 1, 300, 2049, 700, 14, True),
    ("bmm_nt", 3, 100, 70, 130, 13, False),
    ("mm_nt", 1, 1023, 2049, 16384 + 1, 15, True),   # split streams with an extra column
])
def test_unpadded_rows(dev, kind, batch, M, N, K, P, corr):
    _check(dev, kind, batch, M, N, K, P, corr)
