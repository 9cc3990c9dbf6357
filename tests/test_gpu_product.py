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
    ("mm", 1, 40, 24, 600_000, 15, True, True),
    ("mm", 1, 100, 130, 140_001, 15, True, True),   # 128-row plane tiles: two column tiles
    ("bmm", 3, 129, 60, 131_200, 14, False, True),
    ("mm", 1, 3, 2, 1_200_000, 15, True, True),     # past the workspace bound: segmented
    ("mm", 1, 2, 3, 2_096_200, 15, True, True),     # past the whole-K bound: segmented
])
def test_whole_k(dev, kind, batch, M, N, K, P, corr, exact):
    _check(dev, kind, batch, M, N, K, P, corr, exact)


def test_whole_k_other_moduli(dev):
    """A list outside the default one, with an even modulus below 256 (its tie fix), on
    128-row plane tiles."""
    A, B = _pair("mm", 1, 70, 90, 132_000, 3, dev)
    primes = [254, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217]
    got = capi.product("mm", A, B, primes, fill=0x5A)
    ref, _, _ = capi.run("mm", A, B, primes)
    torch.cuda.synchronize()
    assert bits_equal(got.cpu().numpy(), ref.cpu().numpy())


def test_workspace_fallback_takes_the_staged_size(dev):
    """A whole-K product that the allocator cannot give its workspace runs segmented in that
    form's own, not in half of the larger one."""
    import fp64_emu
    M, N, K = 300, 300, 400_000
    A, B = _pair("mm", 1, M, N, K, 5, dev)
    P, corr = fp64_emu.plan_config(K)
    full = capi.product_workspace(1, M, N, K, fp64_emu._PRIMES[:P], corr)
    staged = capi.workspace_size(1, M, N, K, P, corr)
    assert full > 2.5 * staged
    want = fp64_emu.mm(A, B)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held = torch.cuda.memory_reserved()
    total = torch.cuda.get_device_properties(dev).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((held + 0.7 * full) / total, dev)
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        got = fp64_emu.mm(A, B)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert torch.cuda.max_memory_allocated() - before < staged + (64 << 20)
    assert bits_equal(got.cpu().numpy(), want.cpu().numpy())


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


# Whole rounds: single items (fewer than 512 units, or more than 64 k-steps) and item
# streams (512 units and more of at most 64 k-steps) with the correction as two slots, the
# rounds not quite whole, no correction (13 slots), members, ragged edges, both combines.
@pytest.mark.parametrize("kind,batch,M,N,K,P,corr,exact", [
    ("mm_nt", 1, 1000, 1024, 2600, 14, True, True),      # 1 round
    ("mm", 1, 1279, 1500, 2561, 14, True, True),         # 1.9 rounds
    ("bmm_nt", 19, 250, 256, 2700, 13, False, True),     # 247 of 256 units
    ("bmm", 16, 256, 230, 4200, 14, True, False),        # past the streams' depth
    ("mm", 1, 1792, 2000, 1537, 14, True, True),         # 3.5 rounds: staged
    ("mm_nt", 1, 2000, 2000, 2000, 14, True, True),      # streams: 4 rounds of 32 k-steps
    ("mm", 1, 2048, 2030, 3000, 14, True, False),        # of 47
    ("mm_nt", 1, 1000, 4000, 4096, 14, True, True),      # of 64, the most
    ("mm", 1, 1500, 2048, 2300, 14, True, True),         # 3 rounds of 36
    ("bmm_nt", 16, 500, 512, 1536, 14, True, True),      # members, 24 k-steps
    ("bmm", 8, 512, 500, 2100, 14, True, True),          # 2 rounds of 33
])
def test_whole_rounds(dev, kind, batch, M, N, K, P, corr, exact):
    primes = O.PRIMES[:P]
    if corr and batch * (-(-M // 256)) * (-(-N // 256)) * (P + 2) % 256 == 0:   # whole: one corr plane more, or no split
        assert capi.product_workspace(batch, M, N, K, primes) != capi.workspace_size(batch, M, N, K, P, True)
    _check(dev, kind, batch, M, N, K, P, corr, exact)


# On a workspace shorter than it asks for the call runs as the staged entry points do, in
# row chunks where it must: a byte short, the staged size, the minimum, and refused below.
@pytest.mark.parametrize("kind,batch,M,N,K,P", [
    ("mm", 1, 1000, 1024, 1000, 14),         # fused: less than any staged form asks for
    ("mm_nt", 1, 2000, 2048, 3000, 14),      # whole rounds: staged, then chunked
    ("bmm", 16, 512, 512, 1536, 14),         # members: staged, never chunked
    ("mm", 1, 40, 24, 140_000, 15),          # whole K: segmented
    ("mm", 1, 300, 600, 131_072, 15),
])
def test_shorter_workspace(dev, kind, batch, M, N, K, P):
    print(f"case shorter workspace {kind} b={batch} {M}x{N}x{K}", flush=True)
    A, B = _pair(kind, batch, M, N, K, 7, dev)
    primes = O.PRIMES[:P]
    asked = capi.product_workspace(batch, M, N, K, primes, nt=kind.endswith("_nt"))
    staged = capi.workspace_size(batch, M, N, K, P, True)
    least = capi.workspace_size_min(batch, M, N, K, P, True)
    ref, _, _ = capi.run(kind, A, B, primes)
    for size in sorted({asked, asked - 256, asked + 4096, staged, staged - 256, (staged + least) // 2, least}):
        if size >= min(asked, least):
            got = capi.product(kind, A, B, primes, fill=0x5A, ws_bytes=size)
            torch.cuda.synchronize()
            assert bits_equal(got.cpu().numpy(), ref.cpu().numpy()), size
    with pytest.raises(capi.CapiError, match="workspace too small"):
        capi.product(kind, A, B, primes, ws_bytes=min(asked, least) - 256)


# Fused GEMM and reconstruction: each tile (32 x 32, 64 x 32, 64 x 64), edges inside and
# at fragments and tiles, one k-step, depths that are not a multiple of the steps in
# flight, members, both combines, 13 and 14 moduli, with and without the correction.
@pytest.mark.parametrize("kind,batch,M,N,K", [
    ("mm", 1, 1, 1, 1), ("mm_nt", 1, 16, 17, 64), ("mm", 1, 33, 31, 65), ("bmm_nt", 3, 47, 50, 200),
    ("mm_nt", 1, 512, 512, 64 * 17),                                           # 32 x 32, 256 tiles
    ("bmm", 5, 400, 410, 3 * 64 + 5), ("bmm_nt", 40, 129, 200, 257),           # 64 x 32
    ("mm", 1, 800, 900, 700), ("bmm_nt", 12, 500, 300, 500), ("mm_nt", 1, 1025, 1000, 1100),   # 64 x 64 (the last: staged)
    ("mm", 1, 1000, 1024, 2000), ("mm_nt", 1, 1400, 1390, 600),   # 64 x 64 of 32 k-steps; past one round
])
@pytest.mark.parametrize("P,corr,exact", [(14, True, True), (13, False, True), (14, True, False), (13, True, False),
                                          (14, False, True)])
def test_fused(dev, kind, batch, M, N, K, P, corr, exact):
    _check(dev, kind, batch, M, N, K, P, corr, exact)


def test_fused_zero_and_nonfinite(dev):
    """Zeros give +0; rows and columns holding infinities or NaN change only
    what they change in the staged form (their values extract to 0 and the
    width stays at 53 bits)."""
    for special in (0.0, float("inf"), float("-inf"), float("nan"), 1e308, 5e-324):
        print(f"case fused special {special}", flush=True)
        A, B = _pair("mm", 1, 70, 90, 130, 9, dev)
        A[3, 5] = special
        A[7] = 0.0
        B[:, 11] = special
        got = capi.product("mm", A, B, O.PRIMES[:14])
        ref, _, _ = capi.run("mm", A, B, O.PRIMES[:14])
        torch.cuda.synchronize()
        assert bits_equal(got.cpu().numpy(), ref.cpu().numpy())


# Sizing of short rows, eight a wave: rows that end inside a wave's eight and a group's
# 32, one to 320 elements, rows of every scale, an all-zero and an infinite row.
@pytest.mark.parametrize("batch,M,N,K", [(97, 64, 63, 1), (64, 100, 97, 65), (49, 130, 127, 256), (41, 150, 151, 257),
                                         (31, 200, 203, 320)])
def test_short_row_sizing(dev, batch, M, N, K):
    import numpy as np
    from parity_util import oracle_sizing
    print(f"case short rows bmm b={batch} {M}x{N}x{K}", flush=True)
    g = torch.Generator().manual_seed(K)
    A = torch.randn((batch, M, K), dtype=torch.float64, generator=g)
    B = torch.randn((batch, N, K), dtype=torch.float64, generator=g)
    for X in (A, B):
        X *= torch.pow(2.0, torch.randint(-60, 61, X.shape[:2] + (1,), generator=g).double())
    A[3, 5] = 0.0
    B[7, 11, 0] = float("inf")
    assert batch * (M + N) >= 12288
    _, ws, lay = capi.run("bmm", A.to(dev), B.to(dev), O.PRIMES[:14])
    torch.cuda.synchronize()
    gsA, gsB, glA, glB, gbe = capi.sizing(ws[:lay.off_planesA].cpu().numpy(), lay)
    be, sA, sB, lA, lB = oracle_sizing(A.numpy(), B.numpy(), False, O.PRIMES[:14], 53)
    assert gbe == be and np.array_equal(gsA, sA) and np.array_equal(gsB, sB)
    for got, want in ((glA, lA), (glB, lB)):   # float log2-norms: an ulp, rarely (libm's log2)
        off = got != want
        assert off.mean() < 1e-3
        gi, wi = got[off].view(np.int32).astype(np.int64), want[off].view(np.int32).astype(np.int64)
        assert np.all(np.abs(gi - wi) <= 1)
