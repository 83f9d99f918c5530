"""GPU checks of the FP32 matrix kernel for far more lefts than rights: the check of the lefts' values,
made while the few rights are copied, reads every left, and parity with the CPU oracle."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def run(left, right, **kw):
    x = xcorr()
    shape = x.result_shape("n_to_m", left.shape[1], left.shape[2], left.shape[0], right.shape[0])
    out = torch.full(shape, 7.0, device="cuda")
    x.cross_corr("n_to_m", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fp32", **kw)
    torch.cuda.synchronize()
    return out.cpu().numpy(), x.last_launch()["kernel"]


@pytest.mark.parametrize("n,m,rows,cols", [(400, 12, 20, 17), (700, 16, 12, 16)])
def test_the_last_left_is_checked(n, m, rows, cols):
    left, right = seeded((n, rows, cols), "u11", 97, np.float32), seeded((m, rows, cols), "u01", 98, np.float32)
    clean, kernel = run(left, right)
    assert kernel == "direct_pairs_kernel<f32> matrix instructions"
    for k in (0, n - 1):
        l64, r64 = left[k:k + 1].astype(np.float64), right.astype(np.float64)
        err, _ = norm_error(clean[k * m:(k + 1) * m], oracle_family("n_to_m", l64, r64),
                            oracle_family("n_to_m", l64, r64, absval=True))
        assert err <= 1e-6, (n, m, rows, cols, err)
    left[n - 1, rows - 1, cols - 1] = np.nan
    got, _ = run(left, right)
    tiles, _ = run(left, right, tile=1, split=1)
    np.testing.assert_array_equal(got, tiles)
