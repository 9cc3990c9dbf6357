"""CPU tier: the public calls under symbolic-shape tracing (make_fx, fake tensors with a
shape environment, non-strict export): sizes arrive as SymInt, which has no hash."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.fx.experimental.symbolic_shapes import ShapeEnv

import fp64_emu

F64 = torch.float64


@pytest.fixture(autouse=True)
def tables():
    """The kept modulus tables are the trace's own: made in it, and not left to later calls."""
    fp64_emu._tables.cache_clear()
    yield
    fp64_emu._tables.cache_clear()


def _shapes(name, M=40, N=24, K=96):
    b = (3,) if name.startswith("bmm") else ()
    return b + (M, K), b + ((K, N) if name.endswith("_nt") else (N, K))


@pytest.mark.parametrize("name", ["mm", "mm_nt", "bmm", "bmm_nt"])
def test_symbolic_make_fx(name):
    fn = getattr(fp64_emu, name)
    args = [torch.empty(s, dtype=F64, device="meta") for s in _shapes(name)]
    gm = make_fx(lambda A, B: fn(A, B), tracing_mode="symbolic")(*args)
    calls = [n for n in gm.graph.nodes if "fp64_emu_" + name in str(n.target)]
    assert len(calls) == 1 and "sym_size" in gm.code


@pytest.mark.parametrize("name", ["mm", "mm_nt", "bmm", "bmm_nt"])
def test_fake_tensors_of_symbolic_sizes(name):
    real = [torch.empty(s, dtype=F64, device="meta") for s in _shapes(name)]
    with FakeTensorMode(shape_env=ShapeEnv()) as mode:
        args = [mode.from_tensor(t, static_shapes=False) for t in real]
        assert any(isinstance(n, torch.SymInt) for n in args[0].shape)
        out = getattr(fp64_emu, name)(*args)
        want = args[0].shape[:-1] + (args[1].shape[-1 if name.endswith("_nt") else -2],)
        assert tuple(out.shape) == tuple(want) and out.dtype == F64


def test_export_with_dynamic_sizes():
    class Product(torch.nn.Module):
        def forward(self, A, B):
            return fp64_emu.mm(A, B)

    m, k = torch.export.Dim("m", min=2, max=1024), torch.export.Dim.AUTO   # (the plan may pin K)
    with FakeTensorMode():
        A, B = (torch.empty(s, dtype=F64, device="cuda") for s in _shapes("mm"))
    ep = torch.export.export(Product(), (A, B), dynamic_shapes=({0: m, 1: k}, {1: k}), strict=False)
    assert any("fp64_emu_mm" in str(n.target) for n in ep.graph.nodes)
