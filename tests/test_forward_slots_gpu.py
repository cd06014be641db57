"""The forward's slot blocks (8 and 16 receivers, interleaved LDS traces): the
fixed-point sums are exact and do not depend on the order of the adds, so the
data are bitwise those of the blocks of 4 receivers, at every edge of their
range: last blocks of one receiver, traces that just fit or just miss a
workgroup's LDS, tiles shared between workgroups."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import geometry as G

pytestmark = pytest.mark.gpu


def _op(nr, nt, nx=37, nz=29, ns=3, dynamic=False, neg=False, **kw):
    import pylops_amd
    x, z = np.arange(nx) * 10.0, np.arange(nz) * 10.0
    srcs = np.vstack((np.linspace(0, x[-1], ns), np.zeros(ns)))
    recs = np.vstack((np.linspace(0, x[-1], nr) if nr > 1 else [55.0], np.zeros(nr)))
    kw = dict(dict(z=z, x=x, t=np.arange(nt) * 0.004, srcs=srcs, recs=recs, vel=1500.0,
                   wav=G.wav.astype(np.float32), wavcenter=G.wavc, mode="analytic",
                   dynamic=dynamic, dtype="float32"), **kw)
    if neg:
        ts, tr, *_ = pylops_amd.Kirchhoff._traveltime_table(z, x, srcs, recs, 1500.0,
                                                            mode="analytic")
        kw.update(mode="byot", trav=(ts - 0.0113, tr - 0.0087), vel=None)
    return pylops_amd.Kirchhoff(**kw), kw


@pytest.mark.parametrize("nr", [1, 8, 9, 16, 17, 33])
@pytest.mark.parametrize("case", ["kin", "f16", "neg", "dyn", "dyn_gate", "dyn_f16"])
def test_slot_blocks_bitwise(case, nr):
    kw = {}
    if "f16" in case:
        kw["tabledtype"] = "float16"
    if "dyn" in case:
        kw.update(dynamic=True, angleaperture=70)
    if "gate" in case:
        kw["aperture"] = 1.5
    op, okw = _op(nr, 150, neg=case == "neg", **kw)
    m = np.random.default_rng(nr).standard_normal(op.shape[1]).astype(np.float32)
    op.rblock = 4
    want, traces = np.asarray(op @ m), np.asarray(op.spread(m))
    for rb in (8, 16):
        op.rblock = rb
        np.testing.assert_array_equal(op @ m, want, err_msg=str(rb))
        np.testing.assert_array_equal(op.spread(m), traces, err_msg=str(rb))
    if case in ("kin", "dyn", "dyn_gate"):
        # float32 sums against the oracle's float32 operator
        assert G.relerr(want, O.KirchhoffOracle(**okw).matvec(m)) < 1e-5


@pytest.mark.parametrize("nt", [41, 639, 641, 1279, 1281, 2559, 2561])
def test_slot_blocks_trace_lengths(nt):
    """16 slots up to 1280 samples, 8 up to 2560, 4 beyond; one or two
    workgroups per CU."""
    op, _ = _op(19, nt)
    m = np.random.default_rng(nt).standard_normal(op.shape[1]).astype(np.float32)
    op.rblock = 4
    want = np.asarray(op @ m)
    for rb in (8, 16):
        op.rblock = rb
        np.testing.assert_array_equal(op @ m, want, err_msg=str(rb))


@pytest.mark.parametrize("kind", ["finite", "nonfinite", "dyn_f16"])
def test_slot_blocks_shared_tiles(kind):
    """With a workspace the last pairs' tiles are shared by several workgroups
    and their sums added in a second launch: bitwise the same data."""
    import ctypes
    import torch
    from pylops_amd import _lib
    kw = dict(dynamic=True, tabledtype="float16") if kind == "dyn_f16" else {}
    op, _ = _op(45, 300, nx=131, nz=250, ns=2, **kw)
    m = torch.randn(op.shape[1], generator=torch.Generator().manual_seed(1)).cuda()
    if kind == "nonfinite":
        m[1234] = float("inf")
    op.rblock = 4
    want = op @ m
    op.rblock = 16
    L = _lib.load()
    plan = op.plan
    need = L.kx_forward_work_bytes(ctypes.byref(plan))
    base = L.kx_workspace_bytes(ctypes.byref(plan))
    assert need > base  # several workgroups per pair
    for nbytes in (base, need):
        work = torch.empty(nbytes, dtype=torch.uint8, device=m.device)
        d = torch.empty_like(want)
        _lib.check(L.kx_forward_ws(ctypes.byref(plan), _lib.ptr(m), _lib.ptr(d), _lib.ptr(work),
                                   nbytes, _lib.stream_ptr(m.device)))
        if kind == "nonfinite":
            # float64 sums whose order varies: 1e-6 of the largest where finite
            ok = torch.isfinite(want)
            assert torch.equal(ok, torch.isfinite(d))
            assert (d[ok] - want[ok]).abs().max() <= 1e-6 * want[ok].abs().max()
        else:
            assert torch.equal(d, want)
    with pytest.raises(ValueError, match="workspace"):
        _lib.check(L.kx_forward_ws(ctypes.byref(plan), _lib.ptr(m), _lib.ptr(d), _lib.ptr(work),
                                   base - 1, _lib.stream_ptr(m.device)))


def test_forward_leaves_its_workspace_untouched():
    """kx_forward, whose header says so: no tile is shared through it."""
    import ctypes
    import torch
    from pylops_amd import _lib
    op, _ = _op(45, 300, nx=131, nz=250, ns=2)
    m = torch.randn(op.shape[1], generator=torch.Generator().manual_seed(1)).cuda()
    op.rblock = 16
    plan, L = op.plan, _lib.load()
    work = torch.full((L.kx_workspace_bytes(ctypes.byref(plan)),), 7, dtype=torch.uint8,
                      device=m.device)
    d = torch.empty(op.shape[0], device=m.device)
    _lib.check(L.kx_forward(ctypes.byref(plan), _lib.ptr(m), _lib.ptr(d), _lib.ptr(work),
                            _lib.stream_ptr(m.device)))
    assert (work == 7).all()
    assert torch.equal(d, op @ m)
