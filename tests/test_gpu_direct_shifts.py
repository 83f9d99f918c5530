"""GPU parity of the FP32 direct method's 16 x 16 shifts kernel (the default for few rights per
left) against the CPU oracle: edges of its tiles, panels (8 rows x 16 columns) and row shares, one
to four waves per block, and inputs with an infinity or a NaN, which only the shifts whose
overlap holds them may show.  Bar of the FP32 direct method: normalised error <= 1e-6 (products
summed in FP32 partials of at most 64, added in FP64)."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NAME = "direct_kernel<f32> 16x16 shifts"


def run(family, left, right):
    x = xcorr()
    shape = x.result_shape(family, left.shape[1], left.shape[2], left.shape[0], right.shape[0])
    out = torch.full(shape, float("nan"), device="cuda")
    print(f"shifts {family} {left.shape} {right.shape}", flush=True)
    x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fp32")
    torch.cuda.synchronize()
    return out.cpu().numpy(), x.last_launch()["kernel"]


@pytest.mark.parametrize("family,rows,cols,n,m", [
    ("one_to_one", 1, 1, 1, 1), ("one_to_one", 8, 8, 1, 1), ("one_to_one", 9, 16, 1, 1), ("one_to_one", 17, 33, 1, 1),
    ("one_to_many", 19, 20, 1, 5), ("one_to_many", 20, 19, 1, 3), ("one_to_one", 40, 15, 1, 1),
    ("n_to_mn", 33, 31, 2, 6), ("n_to_m", 24, 40, 3, 5), ("one_to_one", 64, 64, 1, 1), ("n_to_m", 100, 60, 2, 3),
    ("one_to_one", 200, 3, 1, 1), ("one_to_one", 5, 80, 1, 1), ("one_to_many", 130, 129, 1, 2)])
def test_parity(family, rows, cols, n, m):
    left = seeded((n, rows, cols), "u01", 41, np.float32)
    right = seeded((m, rows, cols), "u01", 42, np.float32)
    got, kernel = run(family, left, right)
    assert kernel.startswith(NAME)
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(got, oracle_family(family, l64, r64), oracle_family(family, l64, r64, absval=True))
    assert err <= 1e-6, (family, rows, cols, err)


def test_flat_matrices_keep_the_register_tiles():
    left = seeded((1, 5, 81), "u01", 43, np.float32)
    got, kernel = run("one_to_one", left, left)
    assert kernel.startswith("direct_kernel<f32> ty")
    l64 = left.astype(np.float64)
    ref = oracle_family("one_to_one", l64, l64)
    assert norm_error(got, ref, ref)[0] <= 1e-6


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_values_that_are_not_finite_stay_in_their_overlaps(value):
    left = seeded((1, 37, 45), "u01", 44, np.float32)
    right = seeded((2, 37, 45), "u01", 45, np.float32)
    right[1, 30, 2] = value
    left[0, 3, 44] = value
    right[:, :, 7] = 0.0  # inf * 0 inside an overlap is NaN
    got, kernel = run("one_to_many", left, right)
    assert kernel.startswith(NAME)
    with np.errstate(invalid="ignore"):
        ref = oracle_family("one_to_many", left.astype(np.float64), right.astype(np.float64))
    fine = np.isfinite(ref)
    assert (~fine).any() and fine.any()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(got[~fine & ~np.isnan(ref)], ref[~fine & ~np.isnan(ref)].astype(np.float32))
    np.testing.assert_allclose(got[fine], ref[fine], rtol=1e-6)  # positive data: the bar itself
