"""The adjoint of plans whose samples all lie in the staged windows: bitwise
the image of the general kernel, which takes over when the plan's fit bits are
cleared, for every number of tiles per wave and of waves per group, at ragged
tiles, at the first and last samples of a trace, with values that are not
finite; and tables that do not fit keep the general kernel.  (The grids give
every launch shape the workgroup per CU below which the general kernel runs.)"""
import numpy as np
import pytest

from oracle import oracle as O
from tests import geometry as G

pytestmark = pytest.mark.gpu
FIT = 2 | 4 | 8


def _op(ns=5, nr=66, nt=150, nx=517, nz=509, ny=0, dx=1.0, dtype="float32", **kw):
    import pylops_amd
    x, z = np.arange(nx) * dx, np.arange(nz) * dx
    y = np.arange(ny) * dx if ny else None
    line = lambda n: np.linspace(0, x[-1], n) if n > 1 else np.array([55.0])  # noqa: E731
    rows = lambda n: ([np.full(n, 11.0)] if ny else []) + [line(n), np.zeros(n)]  # noqa: E731
    kw = dict(dict(z=z, x=x, y=y, t=np.arange(nt) * 0.004, srcs=np.vstack(rows(ns)),
                   recs=np.vstack(rows(nr)), vel=1500.0, wav=G.wav.astype(dtype),
                   wavcenter=G.wavc, mode="analytic", dtype=dtype), **kw)
    return pylops_amd.Kirchhoff(**kw), kw


def _check(op, d, gt=(1, 2, 4), gs=(1, 2, 4)):
    p = op._plan
    assert p.tabs & FIT == FIT
    for gtiles in gt:
        for gsplit in gs:
            p.gtiles, p.gsplit, tabs = gtiles, gsplit, p.tabs
            got = np.asarray(op.H @ d)
            p.tabs = tabs & ~FIT
            want = np.asarray(op.H @ d)
            p.tabs = tabs
            np.testing.assert_array_equal(got, want, err_msg=f"{gtiles} {gsplit}")
    return got


@pytest.mark.parametrize("case", ["kin", "kin_f16", "kin_f64", "dyn", "dyn_f16", "dyn_f64",
                                  "gate", "gate_f16"])
@pytest.mark.parametrize("ns,nr", [(1, 1), (5, 63), (17, 64), (18, 127)])
def test_fit_bitwise(case, ns, nr):
    kw = {}
    if "f16" in case:
        kw["tabledtype"] = "float16"
    if "f64" in case:
        kw["dtype"] = "float64"
    if "dyn" in case or "gate" in case:
        kw["dynamic"] = True
    if "gate" in case:
        kw.update(aperture=1.5, angleaperture=70)
    op, okw = _op(ns, nr, **kw)
    d = np.random.default_rng(nr).standard_normal(op.shape[0]).astype(op.dtype)
    got = _check(op, d)
    if case in ("kin", "dyn", "gate") and nr < 64:
        # float32 sums against the oracle's float32 operator
        assert G.relerr(got, O.KirchhoffOracle(**okw).rmatvec(d)) < 1e-5
    d[::97] = np.inf
    d[::131] = np.nan
    _check(op, d, gt=(2,), gs=(4,))


@pytest.mark.parametrize("nt", [41, 64, 65, 101])
def test_fit_trace_ends(nt):
    """Windows past both ends of the trace, and traces shorter than a window
    (a table entry past the trace's end would not fit, a sum past it does)."""
    op, _ = _op(3, 20, nt=nt, dx=0.2)
    _check(op, np.random.default_rng(nt).standard_normal(op.shape[0]).astype("float32"))


def test_fit_3d_and_models():
    op, _ = _op(4, 9, nx=65, nz=66, ny=63, dx=2.0)
    _check(op, np.random.default_rng(0).standard_normal(op.shape[0]).astype("float32"))
    import torch
    D = torch.randn(op.shape[0], 7, generator=torch.Generator().manual_seed(2)).cuda()
    tabs = op._plan.tabs
    got = op.H @ D
    op._plan.tabs = tabs & ~FIT
    assert torch.equal(got, op.H @ D)


def test_wide_tables_do_not_fit():
    """Cells of many samples: a tile spans more than a window."""
    op, _ = _op(3, 20, nx=37, nz=29, nt=400, dx=60.0)
    assert op._plan.tabs & FIT == 0


@pytest.mark.parametrize("gsplit,gtiles", [(1, 2), (4, 2), (2, 1)])
@pytest.mark.parametrize("fits", [(1, 1, 1), (1, 0, 1), (0, 0, 0)])
@pytest.mark.parametrize("dynamic", [False, True])
def test_fit_batch_mixed(dynamic, fits, gsplit, gtiles):
    """Problems of a batch that fit beside problems that do not."""
    from pylops_amd.waveeqprocessing import KirchhoffBatch
    ops = [_op(3 + 5 * k, 70 - 21 * k, nx=37 + 8 * k, nz=29, dynamic=dynamic)[0]
           for k in range(3)]
    for op, fit in zip(ops, fits):
        assert op.plan.tabs & FIT == FIT
        if not fit:
            op.plan.tabs &= ~FIT
    B = KirchhoffBatch(ops, gsplit=gsplit, gtiles=gtiles)
    d = np.random.default_rng(1).standard_normal(B.shape[0]).astype("float32")
    got, n, k = np.asarray(B.H @ d), 0, 0
    for op in ops:
        op.gsplit, op.gtiles = B.gsplit, B.gtiles
        want = np.asarray(op.H @ d[k:k + op.shape[0]])
        np.testing.assert_array_equal(got[n:n + op.shape[1]], want)
        n, k = n + op.shape[1], k + op.shape[0]
