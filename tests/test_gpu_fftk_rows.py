"""GPU checks of the own FFT's row kernels where a group of row pairs ends at the matrix: the
row after the last of an odd matrix is padding, whatever lies behind it in memory.
"""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# one size per row kernel: register transforms of 256 points, of 3 * 64 (rows_fwd3)
SIZES = [(129, 100), (151, 65), (65, 90), (35, 200)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows,cols", SIZES)
def test_the_next_matrix_is_not_read_as_padding(rows, cols, dtype):
    """Every second right matrix is NaN: the others' results are those of finite neighbours."""
    x = xcorr()
    left = seeded((1, rows, cols), "normal", 41, dtype)
    right = seeded((4, rows, cols), "u11", 42, dtype)
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    ref = oracle_family("one_to_many", l64, r64)
    scale = oracle_family("one_to_many", l64, r64, absval=True)
    right[1::2] = np.nan
    out = x.cross_corr("one_to_many", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(),
                       precision="fft64", tile=1).cpu().numpy()
    err, _ = norm_error(out[::2], ref[::2], scale[::2])
    assert err <= (1e-6 if dtype is np.float32 else 1e-9), (rows, cols, err)
    assert np.isnan(out[1::2]).all()
