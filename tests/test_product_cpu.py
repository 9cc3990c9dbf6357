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
