"""The tuner's candidates and cache: shapes that the library runs apart, and
entries measured with other kernels are not reused."""
import json

import numpy as np
import pytest

from pylops_amd import _lib
from pylops_amd.waveeqprocessing import autotune as _  # noqa: F401  (the function)
import importlib

A = importlib.import_module("pylops_amd.waveeqprocessing.autotune")
LDS = 160 * 1024


def _cands(*args):
    return list(A._candidates_fwd(*args))


def test_slot_blocks_are_tried_once_each():
    c = _cands("float32", 1280, 400, LDS)
    big = [x for x in c if x[0] > 4]
    # 1280 samples: 16 traces fit (no padding); 8 and 16 ignore the lane order
    # and hold receivers
    assert [x[0] for x in big] == [16, 8]
    assert {x[2] for x in big} == {_lib.KX_SIDE_RECEIVERS}
    assert [x[0] for x in _cands("float32", 1281, 400, LDS) if x[0] > 4] == [8]
    assert not [x for x in _cands("float32", 2561, 400, LDS) if x[0] > 4]
    assert [x[0] for x in _cands("float32", 200, 8, LDS) if x[0] > 4] == [8]
    assert not [x for x in _cands("float64", 200, 400, LDS) if x[0] > 4]


def test_rows_are_tried_in_every_order_and_side():
    c = _cands("float32", 500, 30, LDS)
    assert len(set(c)) == len(c)
    assert {x for x in c if x[0] == 4} == {(4, o, s) for o in A.SORDERS for s in A.SSIDES}
    assert {x[2] for x in _cands("float64", 500, 30, LDS)} == {_lib.KX_SIDE_RECEIVERS}


def _kw():
    x, z, y = np.arange(40) * 10.0, np.arange(40) * 10.0, np.arange(36) * 10.0
    rng = np.random.default_rng(0)
    pts = lambda n: np.vstack((rng.uniform(0, y[-1], n), rng.uniform(0, x[-1], n),  # noqa: E731
                               np.zeros(n)))
    return dict(z=z, x=x, y=y, t=np.arange(400) * 0.004, srcs=pts(6), recs=pts(96), vel=2000.0,
                wav=np.ones(21, np.float32), wavcenter=10, mode="analytic", dtype="float32")


def test_cache_keys_name_the_kernels_and_the_wavelet(monkeypatch):
    monkeypatch.setattr(A.torch.cuda, "get_device_name", lambda dev: "card")
    kw = _kw()
    key = A._key("op", [kw], None)
    assert f"k{A.KERNELS}" in key.split("|")
    assert A._key("op", [dict(kw, wav=np.ones(301, np.float32))], None) != key
    monkeypatch.setattr(A, "KERNELS", A.KERNELS + 1)
    assert A._key("op", [kw], None) != key


@pytest.mark.gpu
def test_entries_of_earlier_kernels_are_measured_again(tmp_path):
    """An entry that fixes blocks of 4, as measured before the slot blocks,
    kept them switched off; on this grid those are about twice as fast."""
    import torch
    kw = _kw()
    g = A._geometry(kw)
    key = (f"op|{torch.cuda.get_device_name(0)}|" + "x".join(str(v) for v in g)
           + ":0:float32:None")
    cache = tmp_path / "tune.json"
    cache.write_text(json.dumps({key: dict(tile=[16, 2, 2], rblock=4, sorder=2, sside=1,
                                           gsplit=4, gtiles=4, ms=1.0)}))
    best = A.autotune(cache=str(cache), reps=3, tiles=((16, 2, 2), (8, 4, 2)), **kw)
    assert best["rblock"] in (8, 16)
    assert len(json.loads(cache.read_text())) == 2
    assert A.autotune(cache=str(cache), **kw) == best
