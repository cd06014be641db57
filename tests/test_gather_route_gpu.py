"""Which gather a plan takes whose samples all lie in the staged windows: the
windowless kernel where it is the faster one, the general kernel where a
launch waits for memory (few sources, few waves); the image is bitwise the
same either way."""
import numpy as np
import pytest
import torch

from pylops_amd import _lib

pytestmark = pytest.mark.gpu
FIT = _lib.KX_TAB_FIT1 | _lib.KX_TAB_FIT2 | _lib.KX_TAB_FIT4


def _op(nx, nz, ns, nr, nt, **kw):
    import pylops_amd
    x, z = np.arange(nx) * 10.0, np.arange(nz) * 10.0
    line = lambda n: np.vstack((np.linspace(0, x[-1], n), np.zeros(n)))  # noqa: E731
    return pylops_amd.Kirchhoff(z=z, x=x, t=np.arange(nt) * 0.004, srcs=line(ns), recs=line(nr),
                                vel=2000.0, wav=np.ones(1, kw.get("dtype", "float32")),
                                wavcenter=0, mode="analytic", **dict(dict(dtype="float32"), **kw))


def _kernels(fn):
    from torch.profiler import ProfilerActivity, profile
    fn()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return " ".join(e.key for e in prof.key_averages())


@pytest.mark.parametrize("shape,kw,windowless", [
    ((581, 394, 2, 240, 1001), {}, False),                     # half the slots: 92 and 111 us
    ((544, 159, 1, 205, 1001), dict(dtype="float64"), False),  # 80 and 100 us
    ((401, 250, 2, 160, 1001), dict(dynamic=True), False),     # 76 and 87 us
    ((313, 368, 3, 117, 1001), {}, False),                     # one pass: 49 and 58 us
    ((313, 368, 9, 117, 1001), {}, True),
    ((581, 394, 12, 60, 1001), dict(dynamic=True), True),
    ((301, 201, 16, 60, 1001), dict(dtype="float64"), True),
])
def test_gather_route(shape, kw, windowless):
    op = _op(*shape, **kw)
    d = torch.randn(op.shape[0], generator=torch.Generator().manual_seed(2)).to(
        device="cuda", dtype=torch.float64 if kw.get("dtype") == "float64" else torch.float32)
    assert op.plan.tabs & FIT
    names = _kernels(lambda: op.gather(d))
    assert "gather" in names
    assert ("gather_fit" in names) == windowless
    image = op.gather(d)
    op.plan.tabs &= ~FIT
    assert torch.equal(op.gather(d), image)
