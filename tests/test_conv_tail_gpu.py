"""The row convolution for every number of taps after the chunks of 32 and 16,
in waves with and without outputs; each output against the extended-precision
sum, within the bound of a sum of nh products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("nt", [2, 64, 255, 257, 530])
@pytest.mark.parametrize("nh", list(range(1, 52, 2)) + [65, 97])
def test_conv_taps_after_the_chunks(dtype, nt, nh):
    import torch
    from pylops_amd.signalprocessing.convolve1d import conv_rows
    rng = np.random.default_rng(nh * 4096 + nt)
    x = rng.standard_normal((3, nt)).astype(dtype)
    h = rng.standard_normal(nh).astype(dtype)
    got = conv_rows(torch.from_numpy(x).cuda(), torch.from_numpy(h).cuda())
    got, c = got.cpu().numpy().astype("longdouble"), (nh - 1) // 2
    hl = h.astype("longdouble")
    for g, xr in zip(got, x.astype("longdouble")):
        bound = (nh + 1) * np.finfo(dtype).eps * np.convolve(abs(xr), abs(hl))[c:c + nt]
        assert (abs(g - np.convolve(xr, hl)[c:c + nt]) <= bound).all()
