"""GPU parity of the own FFT where its rows have 48 and 96 points, whose blocks write several output rows
at once: widths at both ends of these lengths, heights that end inside a block; float and double data."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype,tol", [(np.float32, 1e-6), (np.float64, 1e-12)])
@pytest.mark.parametrize("rows,cols", [(257, 17), (300, 24), (129, 18), (150, 33), (131, 48), (260, 40)])
def test_parity(rows, cols, dtype, tol):
    left, right = seeded((1, rows, cols), "u11", 61, dtype), seeded((3, rows, cols), "u01", 62, dtype)
    x = xcorr()
    out = torch.full(x.result_shape("one_to_many", rows, cols, 1, 3), float("nan"), device="cuda",
                     dtype=torch.from_numpy(left).dtype)
    x.cross_corr("one_to_many", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out,
                 precision="fft64", tile=1)
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"] == "fftk_rows_inv"
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(out.cpu().numpy(), oracle_family("one_to_many", l64, r64),
                        oracle_family("one_to_many", l64, r64, absval=True))
    assert err <= tol, (rows, cols, err)
