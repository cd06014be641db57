"""A 2D grid's eikonal sweeps in one launch (kx_eikonal_ws with its
workspace) against one launch per anti-diagonal (kx_eikonal): the same cells
in the same order, so the same rounds and times to rounding."""
import ctypes

import numpy as np
import pytest
import torch

from pylops_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(1, 1), (1, 9), (2, 70), (64, 65), (65, 64), (129, 40),
                                   (40, 130), (1023, 31), (1025, 33), (33, 1030)])
@pytest.mark.parametrize("order", [1, 2])
def test_one_launch_matches_diagonals(nx, nz, order):
    L = _lib.load()
    rng = np.random.default_rng(nx * 1000 + nz)
    n = 35  # past one 32-wide transpose tile
    slow = 1.0 / (1500.0 + 1500.0 * rng.random((nx, nz)))
    slow = torch.as_tensor(slow.ravel(), device="cuda")
    cells = np.zeros((n, 3), np.int32)
    cells[:, 0], cells[:, 2] = rng.integers(0, nx, n), rng.integers(0, nz, n)
    cells[0] = 0
    cells[1] = (nx - 1, 0, nz - 1)
    src = torch.as_tensor(cells, device="cuda")
    need = L.kx_eikonal_work_bytes(2, nx, 1, nz, n)
    assert need >= nx * nz * n * 8
    work = torch.empty(need, dtype=torch.uint8, device="cuda")
    out = []
    for w in (None, work):
        T = torch.empty((nx * nz, n), dtype=torch.float64, device="cuda")
        flag = torch.zeros(1, dtype=torch.int32, device="cuda")
        it = (ctypes.c_int32 * 2)(0, 0)
        _lib.check(L.kx_eikonal_ws(2, nx, 1, nz, 10.0, 1.0, 8.0, _lib.ptr(slow), n, _lib.ptr(src),
                                   _lib.ptr(T), 60, order, _lib.ptr(flag), it,
                                   None if w is None else _lib.ptr(w), 0 if w is None else need,
                                   _lib.stream_ptr(T.device)))
        out.append((T.cpu().numpy(), tuple(it)))
    assert out[0][1] == out[1][1] and out[0][1][1] == 1
    # a round ends when nothing changes by more than 1e-13: the bar of the
    # comparison with the oracle
    np.testing.assert_allclose(out[1][0], out[0][0], rtol=1e-12, atol=0)


def test_no_workspace_for_other_grids():
    L = _lib.load()
    assert L.kx_eikonal_work_bytes(3, 20, 20, 20, 4) == 0
    assert L.kx_eikonal_work_bytes(2, 1100, 1, 1025, 4) == 0
    assert L.kx_eikonal_work_bytes(2, 1100, 1, 1024, 4) > 0
