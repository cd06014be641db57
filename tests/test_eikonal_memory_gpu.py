"""Memory of the one-launch eikonal sweeps: a bounded workspace, tables solved
in groups where it holds fewer of them, and none where nothing is left."""
import ctypes

import numpy as np
import pytest
import torch

from pylops_amd import _lib
from pylops_amd.waveeqprocessing import _tables as T

pytestmark = pytest.mark.gpu
NX, NZ, N = 61, 44, 70


def _solve(work):
    L = _lib.load()
    rng = np.random.default_rng(3)
    slow = torch.as_tensor(1.0 / (1500.0 + 1500.0 * rng.random(NX * NZ)), device="cuda")
    cells = np.zeros((N, 3), np.int32)
    cells[:, 0], cells[:, 2] = rng.integers(0, NX, N), rng.integers(0, NZ, N)
    src = torch.as_tensor(cells, device="cuda")
    out = torch.full((NX * NZ, N), float("nan"), dtype=torch.float64, device="cuda")
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    it = (ctypes.c_int32 * 2)(0, 0)
    _lib.check(L.kx_eikonal_ws(2, NX, 1, NZ, 10.0, 1.0, 8.0, _lib.ptr(slow), N, _lib.ptr(src),
                               _lib.ptr(out), 60, 2, _lib.ptr(flag), it,
                               _lib.ptr(work) if work.numel() else None, work.numel(),
                               _lib.stream_ptr(out.device)))
    return out, tuple(it)


@pytest.mark.parametrize("held", [1, 7, 32, 69, 70])
def test_tables_in_groups(held):
    need = _lib.load().kx_eikonal_work_bytes(2, NX, 1, NZ, held)
    assert need == NX * NZ * held * 8 + 64
    guard = torch.full((need + 4096,), 85, dtype=torch.uint8, device="cuda")
    full, rounds = _solve(torch.empty(_lib.load().kx_eikonal_work_bytes(2, NX, 1, NZ, N),
                                      dtype=torch.uint8, device="cuda"))
    got, it = _solve(guard[:need])
    assert torch.equal(got, full) and it == rounds
    assert bool((guard[need:] == 85).all())


def test_workspace_is_bounded():
    need = _lib.load().kx_eikonal_work_bytes
    assert need(2, 1000, 1, 1000, 4000) == need(2, 1000, 1, 1000, 512)


def test_tables_without_memory_for_a_workspace(monkeypatch):
    x, z = np.arange(40) * 10.0, np.arange(30) * 10.0
    pts = np.vstack((np.linspace(0, x[-1], 90), np.zeros(90)))
    args = (pts, 1500.0 + np.arange(1200.0).reshape(40, 30), np.zeros(2), np.full(2, 10.0),
            np.array([40, 30]), torch.device("cuda"))
    want = T.eikonal(*args)
    empty, sizes = torch.empty, []

    def short(*a, **kw):
        if kw.get("dtype") == torch.uint8 and a[0] > limit:
            sizes.append(a[0])
            raise torch.OutOfMemoryError("no memory for the test")
        return empty(*a, **kw)

    monkeypatch.setattr(torch, "empty", short)
    for limit in (90 * 9600, 0):  # half of the tables, none
        torch.testing.assert_close(T.eikonal(*args), want, rtol=1e-12, atol=0)
    assert len(sizes) >= 2
