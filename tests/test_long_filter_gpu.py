"""Forwards with long filters: the operator spreads and convolves in two
launches where that is faster; the data are those of the convolution in the
spread launch, bitwise."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests import geometry as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntaps", [41, 711])
@pytest.mark.parametrize("tab", [None, "float16"])
def test_long_filters_take_a_launch_of_their_own(ntaps, tab):
    import pylops_amd
    import torch
    from pylops_amd import _lib
    x, z = np.arange(201) * 10.0, np.arange(150) * 10.0
    rng = np.random.default_rng(ntaps)
    kw = dict(z=z, x=x, t=np.arange(751) * 0.004,
              srcs=np.vstack((np.linspace(0, x[-1], 21), np.zeros(21))),
              recs=np.vstack((np.linspace(0, x[-1], 101), np.zeros(101))), vel=1500.0,
              wav=rng.standard_normal(ntaps).astype(np.float32), wavcenter=ntaps // 2,
              mode="analytic", dtype="float32", tabledtype=tab)
    op = pylops_amd.Kirchhoff(**kw)
    m = torch.randn(op.shape[1], generator=torch.Generator().manual_seed(1)).cuda()
    plan, L, st = op.plan, _lib.load(), _lib.stream_ptr(m.device)
    d, e = (torch.empty(op.shape[0], device=m.device) for _ in range(2))
    work = torch.full((op.shape[0],), float("nan"), device=m.device)
    _lib.check(L.kx_forward(ctypes.byref(plan), _lib.ptr(m), _lib.ptr(d), _lib.ptr(work), st))
    _lib.check(L.kx_forward_noalloc(ctypes.byref(plan), _lib.ptr(m), _lib.ptr(e), st))
    assert torch.equal(d, e)
    assert torch.equal(op @ m, d)
    # two launches: the traces pass through the workspace
    assert bool(torch.isnan(work).all()) == (ntaps < 100)
    if ntaps > 100:
        assert torch.equal(work, op.spread(m).reshape(-1))
    if tab is None:
        want = O.KirchhoffOracle(**{k: v for k, v in kw.items() if k != "tabledtype"}).matvec(
            m.cpu().numpy())
        assert G.relerr(d.cpu().numpy(), want) < 1e-5
