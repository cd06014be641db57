"""The forward's choice between blocks of 8 and 16 receivers, whose tiles may
be shared by several workgroups, and the blocks of 4, 2 and 1 (asked
of the library, which reads the card's compute units and LDS)."""
import ctypes

import pytest

from pylops_amd import _lib
from pylops_amd.waveeqprocessing import _tables as T

pytestmark = pytest.mark.gpu


def _plan(nx, ny, nz, ns, nr, nt, dynamic, fmt, nh=81):
    p = T.make_geom_plan(nx, ny, nz, T.default_tile(2 if ny == 1 else 3, nz))
    p.dtype, p.tab_fmt, p.tabs = _lib.KX_F32, fmt, _lib.KX_TAB_SLOTS
    p.dynamic = _lib.KX_DYNAMIC_NOGATE if dynamic else 0
    p.ns, p.nr, p.nt, p.nh = ns, nr, nt, nh
    for k in ("off_s", "base_s", "off_r", "base_r", "wp_s", "wq_s", "wp_r", "wq_r", "izmin",
              "h", "hstar", "aux"):
        setattr(p, k, 16)  # never dereferenced
    return p


def _shared(*args, **kw):
    p, L = _plan(*args, **kw), _lib.load()
    need = L.kx_forward_work_bytes(ctypes.byref(p))
    base = L.kx_workspace_bytes(ctypes.byref(p))
    assert base > 0
    return need > base


@pytest.mark.parametrize("args", [
    # measured: blocks of 4 and the shared slots that an earlier estimate took
    (111, 1, 274, 7, 4, 2379, False, _lib.KX_F32),   # 41 and 71 us
    (158, 1, 184, 1, 5, 1121, False, _lib.KX_F32),   # 29 and 60 us
    (199, 1, 186, 1, 55, 2093, False, _lib.KX_F32),  # 34 and 69 us
    (182, 1, 252, 1, 12, 1387, False, _lib.KX_F32),  # 41 and 81 us
])
def test_few_workgroups_stay_in_blocks_of_4(args):
    assert not _shared(*args)


@pytest.mark.parametrize("args", [
    (32, 32, 40, 2, 9, 251, False, _lib.KX_F32),     # 67 and 27 us
    (301, 1, 200, 5, 33, 1301, True, _lib.KX_F32),   # 101 and 56 us
    (40, 36, 50, 4, 37, 1301, False, _lib.KX_F16),   # 123 and 77 us
])
def test_small_grids_that_gain_share_their_tiles(args):
    assert _shared(*args)
