"""GPU parity of the normalised FFT entry point on float data (the own FP64 FFT up to 2048 rows
and columns, rocFFT beyond) against the CPU oracle: normalised error <= 1e-6 for both values of
fp64_transform, low-overlap corners included, and on both sides of the size limit."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("family,rows,cols,n,m", [("one_to_one", 1, 1, 1, 1), ("one_to_many", 65, 31, 1, 3),
                                                  ("n_to_mn", 40, 70, 2, 4), ("n_to_m", 20, 24, 3, 4),
                                                  ("one_to_one", 3, 2048, 1, 1), ("one_to_one", 2048, 3, 1, 1)])
def test_normalised_float(family, rows, cols, n, m, fp64):
    left = seeded((n, rows, cols), "u01", 31, np.float32)
    right = seeded((m, rows, cols), "u11", 32, np.float32)
    x = xcorr()
    got = x.fft_cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), fp64_transform=fp64)
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"].startswith("fftk")
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(got.cpu().numpy(), oracle_family(family, l64, r64), oracle_family(family, l64, r64, absval=True))
    assert err <= 1e-6, (family, rows, cols, err)


def test_beyond_the_own_fft():
    left = seeded((1, 2, 2049), "u01", 33, np.float32)
    right = seeded((1, 2, 2049), "u01", 34, np.float32)
    x = xcorr()
    got = x.fft_cross_corr("one_to_one", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(),
                           fp64_transform=True)
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"] == "fft_hadamard"
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    ref = oracle_family("one_to_one", l64, r64)
    assert norm_error(got.cpu().numpy(), ref, oracle_family("one_to_one", l64, r64, absval=True))[0] <= 1e-6
