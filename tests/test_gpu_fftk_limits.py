"""GPU checks of the own FFT's one-block kernels at the limits of a call: more pairs than one launch
holds threads for, and batches whose padded spectra would take many times the memory of the
three-pass layout."""
import numpy as np
import pytest

from xc_testutil import seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_more_pairs_than_one_launch_holds():
    """8192 x 8193 pairs of 1x1: 64 threads each are more than 2^32.  A result is one product."""
    x = xcorr()
    left = seeded((8192, 1, 1), "normal", 1, np.float32)
    right = seeded((8193, 1, 1), "normal", 2, np.float32)
    dl, dr = torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda()
    out = torch.full((8192 * 8193, 1, 1), float("nan"), device="cuda")
    print("8192 x 8193 of 1x1", flush=True)
    x.cross_corr("n_to_m", dl, dr, out=out, precision="fft64", tile=1)
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"] == "fftk_small_pairs"
    got = out.view(8192, 8193).double()
    ref = dl.view(-1, 1).double() * dr.view(1, -1).double()
    assert ((got - ref).abs() <= 1e-6 * ref.abs()).all()
