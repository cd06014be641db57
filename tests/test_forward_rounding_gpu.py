"""How far a float32 forward's fixed-point sums lie from the exact ones.  Every
contribution is rounded by at most 2^-31 of the bound 2^ex on the largest
(2^ex the power of two above 2 max|m| wamp), whichever of its two samples it
goes to, and the float32 products before it and the sum after it by 2^-24 of
themselves.

Each image point has two samples of its own here, traveltimes are exact in
float32, and one point is 300 times the others: the rounding is seen alone.
Bar: 2^-31 2^ex, plus 2^-24 of the largest of the other contributions (2^-8)
for each of the three float32 roundings."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NX, NZ, DT = 20, 17, 2.0 ** -8
NT = 2 * NX * NZ + 8


def _problem():
    import pylops_amd
    rng = np.random.default_rng(5)
    ni = NX * NZ
    frac = rng.integers(1, 64, ni) / 64.0
    tr = np.stack([(2 * rng.permutation(ni) + 2 + frac) * DT for _ in range(19)], 1)
    ts = np.zeros((ni, 1))
    x, z = np.arange(NX) * 10.0, np.arange(NZ) * 10.0
    srcs = np.array([[55.0], [0.0]])
    recs = np.vstack((np.linspace(0, x[-1], 19), np.zeros(19)))
    kw = dict(z=z, x=x, t=np.arange(NT) * DT, srcs=srcs, recs=recs, vel=None,
              wav=np.ones(1, np.float32), wavcenter=0, mode="byot", trav=(ts, tr),
              dtype="float32")
    m = rng.uniform(2.0 ** -9, 2.0 ** -8, ni) * rng.choice([-1.0, 1.0], ni)
    m = m.astype(np.float32)
    m[7] = 1.0
    q = tr / DT
    it = q.astype(int)
    want = np.zeros((19, NT))
    for j in range(19):
        f = q[:, j] - it[:, j]
        np.add.at(want[j], it[:, j], m * (1.0 - f))
        np.add.at(want[j], it[:, j] + 1, m * f)
    return pylops_amd.Kirchhoff(**kw), m, want


def _check(d, want):
    ex = 2  # 2 max|m| wamp = 2 < 2^2
    err = np.abs(np.asarray(d, np.float64).reshape(want.shape) - want)
    assert err.max() <= 2.0 ** (ex - 31) + 3 * 2.0 ** -32, err.max() * 2.0 ** 31


@pytest.mark.parametrize("rblock", [1, 4, 8, 16])
def test_contributions_round_by_half_a_unit(rblock):
    op, m, want = _problem()
    op.rblock = rblock
    _check(op.spread(m), want)
    _check(op @ m, want)


def test_contributions_of_models_and_batches_round_alike():
    import torch
    from pylops_amd.waveeqprocessing import KirchhoffBatch
    op, m, want = _problem()
    M = torch.as_tensor(np.stack([m, m * 0.5, -m, m], 1)).cuda()
    D = op.matmat(M).cpu().numpy()
    _check(D[:, 0], want)
    _check(D[:, 1] * 2, want)
    _check(-D[:, 2], want)
    _check(KirchhoffBatch([op]) @ m, want)
