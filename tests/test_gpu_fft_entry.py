"""GPU parity of the normalised FFT entry point on float data (the own FP64 FFT up to 2048 rows
and columns, rocFFT beyond) against the CPU oracle: normalised error <= 1e-6 for both values of
fp64_transform, low-overlap corners included, and on both sides of the size limit."""
import numpy as np
import pytest

from xc_testutil import norm_error, normalize_fft, oracle_family, seeded, xcorr

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


def well_overlapped(rows, cols):
    """Shifts with at least a quarter of the pixels in common.  FP32 transforms leave about 1.5e-7 of
    the results' 2-norm at every shift, which for values in [0, 1) is up to 2e-6 of a sum here."""
    dy = np.abs(np.arange(-(rows - 1), rows))[:, None]
    dx = np.abs(np.arange(-(cols - 1), cols))[None, :]
    return (rows - dy) * (cols - dx) * 4 >= rows * cols


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("rows,cols", [(6, 2049), (2049, 6)])
def test_rocfft_transforms_normalised(rows, cols, fp64):
    left = seeded((1, rows, cols), "u01", 35, np.float32)
    right = seeded((2, rows, cols), "u01", 36, np.float32)
    x = xcorr()
    got = x.fft_cross_corr("one_to_many", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(),
                           fp64_transform=fp64).cpu().numpy()
    assert x.last_launch()["kernel"] == "fft_hadamard"
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err = np.abs(got - oracle_family("one_to_many", l64, r64)) / oracle_family("one_to_many", l64, r64, absval=True)
    print(rows, cols, fp64, err.max(), err[:, well_overlapped(rows, cols)].max())
    assert err[:, well_overlapped(rows, cols)].max() <= (2e-7 if fp64 else 2e-6)
    if fp64:
        assert err.max() <= 1e-6


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("family,rows,cols,n,m", [("one_to_one", 64, 64, 1, 1), ("n_to_m", 16, 12, 3, 4),
                                                  ("n_to_mn", 20, 25, 2, 4)])
def test_unnormalised_float(family, rows, cols, n, m, fp64):
    """The 2H x 2W layout of float data, brought to the definition's by the oracle's reordering."""
    left = seeded((n, rows, cols), "u01", 37, np.float32)
    right = seeded((m, rows, cols), "u01", 38, np.float32)
    x = xcorr()
    raw = x.fft_cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), normalize=False,
                           fp64_transform=fp64).cpu().numpy()
    assert x.last_launch()["kernel"] == "fft_hadamard"
    assert raw.dtype == np.float32 and raw.shape[1:] == (2 * rows, 2 * cols)
    got = np.stack([normalize_fft(r) for r in raw])
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err = np.abs(got - oracle_family(family, l64, r64)) / oracle_family(family, l64, r64, absval=True)
    print(family, rows, cols, fp64, err.max(), err[:, well_overlapped(rows, cols)].max())
    assert err[:, well_overlapped(rows, cols)].max() <= (2e-7 if fp64 else 2e-6)
    if fp64:
        assert err.max() <= 1e-6
