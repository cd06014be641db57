"""Memory of the slot-ordered receiver tables and of the products' workspaces:
the copies exist only where a forward reads them and memory is plentiful, and
products run with the least workspace where more is not to be had."""
import numpy as np
import pytest
import torch

from tests import geometry as G

pytestmark = pytest.mark.gpu


def _op(nx=64, nz=60, ns=3, nr=64, nt=400, ny=0, **kw):
    import pylops_amd
    x, z = np.arange(nx) * 10.0, np.arange(nz) * 10.0
    rng = np.random.default_rng(1)
    if ny:
        y = np.arange(ny) * 10.0
        pts = lambda n: np.vstack((rng.uniform(0, y[-1], n), rng.uniform(0, x[-1], n),  # noqa: E731
                                   np.zeros(n)))
        kw["y"] = y
    else:
        pts = lambda n: np.vstack((np.linspace(0, x[-1], n), np.zeros(n)))  # noqa: E731
    return pylops_amd.Kirchhoff(z=z, x=x, t=np.arange(nt) * 0.004, srcs=pts(ns), recs=pts(nr),
                                vel=2000.0, wav=G.wav.astype(kw.get("dtype", "float32")),
                                wavcenter=G.wavc, mode="analytic",
                                **dict(dict(dtype="float32"), **kw))


def _copied(op):
    """Whether a receiver table's buffer holds more than the table."""
    names = ("off_r", "wp_r", "wq_r") if op.dynamic else ("off_r",)
    more = {op._dev_tables[k].untyped_storage().nbytes() > op._dev_tables[k].nbytes
            for k in names}
    assert len(more) == 1
    return more.pop()


@pytest.mark.parametrize("kw", [
    dict(ny=48, nz=50, sside=2),          # blocks of sources
    dict(ny=48, nz=50, nt=2601),          # 8 traces do not fit LDS
    dict(ny=48, nz=50, rblock=4),
    dict(nx=101, nz=100, ns=11, nr=51),   # blocks of 4 are faster
    dict(ny=48, nz=50, dtype="float64"),
])
def test_tables_that_no_forward_reads_are_not_copied(kw):
    assert not _copied(_op(**kw))


@pytest.mark.parametrize("kw", [dict(ny=48, nz=50), dict(ny=48, nz=50, tabledtype="float16"),
                                dict(nx=301, nz=200, ns=31, nr=121, dynamic=True)])
def test_copies_need_plenty_of_memory(kw, monkeypatch):
    """Without the copies the data are bitwise the same."""
    op = _op(**kw)
    assert _copied(op)
    m = torch.randn(op.shape[1], generator=torch.Generator().manual_seed(1)).cuda()
    total = torch.cuda.mem_get_info()[1]
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev=None: (total // 2, total))
    plain = _op(**kw)
    assert not _copied(plain)
    plain.rblock = 16  # asks for them again, in vain
    assert not _copied(plain)
    assert torch.equal(plain @ m, op @ m)


def test_a_block_size_set_later_brings_the_copies():
    from pylops_amd.waveeqprocessing import KirchhoffBatch
    op = _op(rblock=4, dynamic=True)
    assert not _copied(op)
    batch = KirchhoffBatch([op])
    m = torch.randn(op.shape[1], generator=torch.Generator().manual_seed(2)).cuda()
    d, b = op @ m, batch @ m
    op.rblock = 16
    assert _copied(op)
    assert torch.equal(op @ m, d)
    junk = torch.full((1 << 22,), float("nan"), device="cuda")  # over freed tables
    assert torch.equal(batch @ m, b)
    del junk


def test_adjoints_take_the_traces_alone():
    op = _op(ny=48, nz=50)
    plan = op.plan
    assert op._work_bytes(plan) > op._trace_bytes()  # the forward shares tiles
    d = torch.randn(op.shape[0], generator=torch.Generator().manual_seed(3)).cuda()
    op.H @ d
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    op.H @ d
    peak = torch.cuda.max_memory_allocated() - before
    assert peak <= 4 * (op.shape[0] + op.shape[1]) + 4096


@pytest.mark.parametrize("into", [False, True])
def test_products_run_with_the_least_workspace(into, monkeypatch):
    op = _op(ny=48, nz=50)
    m = torch.randn(op.shape[1], generator=torch.Generator().manual_seed(4)).cuda()
    want = op @ m
    low = _op(ny=48, nz=50)
    monkeypatch.setattr(type(low), "_work_bytes", lambda self, plan: 1 << 46)
    got = torch.empty_like(want)
    if into:
        low._into(m, got, False)
        low._into(m, got, False)
    else:
        got = low @ m
    assert torch.equal(got, want)
