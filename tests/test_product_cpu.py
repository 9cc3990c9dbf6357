"""CPU tier: what fp64emu_product chooses for a call and what it asks of its caller, by its
workspace query and its refusals (no GPU is touched).  A fused product keeps no residue or
correction planes, so it asks for less than the staged layout; a whole-K or whole-rounds one
for more."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
fp64_emu = pytest.importorskip("fp64_emu")
from fp64_emu import capi  # noqa: E402

EINVAL = 1


def _fused(batch, M, N, K, P=14, corr=True):
    return (capi.product_workspace(batch, M, N, K, fp64_emu._PRIMES[:P], corr)
            < capi.workspace_size(batch, M, N, K, P, corr))


def _refusal(batch, M, N, K, P=14, corr=True):
    """The message a call with a full workspace is refused with, "" if it gets to its first
    launch (which fails here, without a device, before any operand is read)."""
    pr = np.asarray(fp64_emu._PRIMES[:P], np.int32)
    p = capi.Product(0x1000, 0x1000, 0x1000, batch, M, N, K, 0, pr.ctypes.data, P, 1, 53, int(corr))
    ws = capi.lib().fp64emu_product_workspace(ctypes.byref(p))
    st = capi.lib().fp64emu_product(ctypes.byref(p), ctypes.c_void_p(0x2000), ws, None)
    return capi.lib().fp64emu_last_error().decode() if st == EINVAL else ""


@pytest.mark.skipif(torch.cuda.is_available(), reason="calls with dummy pointers: only without a GPU")
@pytest.mark.parametrize("batch,M,N,K,fused,refused", [
    (1, 95_000, 95_000, 64, True, False),       # 64 x 32 tiles: 0.53 of a dispatch
    (1, 131_072, 131_008, 64, True, False),     # the last column tile under the bound
    (1, 131_072, 131_072, 64, False, True),     # past it, as the staged form's reconstruction is
    (2_500_000, 65, 64, 64, False, True),       # 10 000 000 groups of 512 threads; staged, too many GEMM groups
])
def test_fused_groups_at_the_dispatch_bound(batch, M, N, K, fused, refused):
    assert _fused(batch, M, N, K) == fused
    assert _refusal(batch, M, N, K) == ("problem too large for one launch" if refused else "")


# Past K = 131071: planes of the whole depth, where they are few times the operands or the
# segmented form's workspace; otherwise the segmented form and no more than it takes.
@pytest.mark.parametrize("batch,M,N,K,whole", [
    (1, 300, 200, 200_000, True), (1, 2000, 2000, 150_000, True), (1, 20, 20, 600_000, True),
    (1, 300, 300, 800_000, True), (1, 129, 300, 131_072, True), (8, 100, 100, 140_000, True),
    (1, 1, 1, 2_000_000, False), (1, 20, 20, 700_000, False), (1, 30, 30, 1_000_000, False),
    (1, 20_000, 64, 140_000, False), (1, 2, 3, 2_096_200, False),
])
def test_whole_k_workspace_is_bounded(batch, M, N, K, whole):
    P, corr = fp64_emu.plan_config(K)
    asked = capi.product_workspace(batch, M, N, K, fp64_emu._PRIMES[:P], corr)
    segmented = capi.workspace_size(batch, M, N, K, P, corr)
    assert (asked > segmented) == whole and asked >= segmented
    assert asked <= max(segmented, min(24 << 30, 5 * max(8 * batch * (M + N) * K, segmented)))


def test_whole_k_planes_hold_the_rows_that_are_read():
    """128 x 128 tiles: planes of 128-row tiles, not 256."""
    M, N, K, P = 100, 30, 200_000, 15
    planes = 2 * 128 * (P + 2) * (-(-K // 64) * 64)
    asked = capi.product_workspace(1, M, N, K, fp64_emu._PRIMES[:P])
    assert planes < asked < 1.1 * planes


def test_whole_k_workspace_fuzz():
    """Seeded shapes and modulus counts of every depth past 131071, the correction on and off."""
    rng = np.random.default_rng(5)
    for _ in range(1500):
        batch = int(np.exp(rng.uniform(0, np.log(50)))) if rng.random() < 0.3 else 1
        M, N = (int(np.exp(rng.uniform(0, np.log(5000)))) for _ in range(2))
        K = int(np.exp(rng.uniform(np.log(131072), np.log(128 * 65536))))
        P, corr = int(rng.integers(1, 21)), bool(rng.integers(2))
        asked = capi.product_workspace(batch, M, N, K, fp64_emu._PRIMES[:P], corr)
        segmented = capi.workspace_size(batch, M, N, K, P, corr)
        bound = max(segmented, min(24 << 30, 5 * max(8 * batch * (M + N) * K, segmented)))
        assert asked <= bound, (batch, M, N, K, P, corr)


# Where fused products lost to the staged form, and where they gain (14 and 13 moduli:
# with the correction and without; the columns are whether the call runs fused).
@pytest.mark.parametrize("batch,M,N,K,with_corr,without", [
    (1, 64, 64, 64, True, True), (1, 333, 501, 777, True, True), (1, 512, 512, 512, True, True),
    (1, 1024, 1024, 1024, True, True), (64, 256, 256, 256, True, True), (1, 4000, 4000, 256, True, True),
    (64, 64, 64, 2560, True, True), (1, 1000, 1000, 2048, True, True),
    (1, 640, 640, 1536, False, False), (1, 480, 500, 3500, False, False), (8, 200, 200, 2048, False, False),
    (24, 128, 128, 2048, False, False), (5, 221, 216, 3776, False, False), (1, 960, 960, 2048, False, False),
    (6, 448, 320, 1984, False, False), (25, 120, 120, 1536, False, False),
    (1, 768, 768, 768, True, False), (1, 2000, 2000, 512, True, False),
])
def test_fused_only_where_it_pays(batch, M, N, K, with_corr, without):
    assert _fused(batch, M, N, K, 14, True) == with_corr
    assert _fused(batch, M, N, K, 13, False) == without


# Whole rounds (the correction as two slots) where they gain, the staged form elsewhere:
# many tiles, a long K-split against rounds not quite whole, few k-steps.
@pytest.mark.parametrize("batch,M,N,K,rounds", [
    (1, 1024, 1024, 2560, True), (1, 2048, 2048, 3000, True), (1, 2000, 2000, 2000, True),
    (16, 512, 512, 8192, True), (16, 512, 512, 1536, True), (8, 512, 512, 2048, True),
    (1, 3072, 3072, 4096, True), (1, 1280, 1536, 4096, True), (1, 4096, 3840, 2000, True),
    (1, 3500, 3500, 2560, False), (1, 3840, 3840, 2600, False), (1, 4096, 3840, 4096, False),
    (1, 1280, 1536, 8192, False), (1, 1280, 1536, 32768, False),
    (1, 1000, 4000, 1536, False), (1, 1024, 2048, 2048, False),
])
def test_whole_rounds_only_where_they_pay(batch, M, N, K, rounds):
    asked = capi.product_workspace(batch, M, N, K, fp64_emu._PRIMES[:14])
    assert (asked != capi.workspace_size(batch, M, N, K, 14, True)) == rounds
