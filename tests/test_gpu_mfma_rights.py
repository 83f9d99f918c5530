"""GPU parity of the split-precision methods' kernel for many rights per left (the default there) against
the CPU oracle: partial groups of 64 rights, tiles of 4 dy x 32 dx that cross the result's edges,
steps of 16 columns that cross the matrix's, odd numbers of right rows per wave, every family; data
that is not finite.  Bar of both methods: normalised error <= 2e-6."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def run(family, left, right, prec, **kw):
    x = xcorr()
    shape = x.result_shape(family, left.shape[1], left.shape[2], left.shape[0], right.shape[0])
    out = torch.full(shape, float("nan"), device="cuda")
    print(f"rights {prec} {family} {left.shape} {right.shape}", flush=True)
    x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision=prec, **kw)
    torch.cuda.synchronize()
    return out.cpu().numpy(), x.last_launch()["kernel"]


@pytest.mark.parametrize("prec", ["bf16x3", "fp16x3"])
@pytest.mark.parametrize("family,rows,cols,n,m", [
    ("one_to_many", 16, 16, 1, 64), ("one_to_many", 33, 32, 1, 33), ("n_to_m", 17, 31, 3, 60),
    ("n_to_mn", 33, 47, 3, 180), ("one_to_many", 64, 64, 1, 64), ("one_to_many", 65, 67, 1, 48),
    ("one_to_many", 301, 1, 1, 64), ("n_to_m", 24, 90, 2, 112), ("n_to_mn", 48, 97, 2, 128),
    ("one_to_many", 130, 20, 1, 128)])
def test_parity(prec, family, rows, cols, n, m):
    left = seeded((n, rows, cols), "u01", 71, np.float32)
    right = seeded((m, rows, cols), "normal", 72, np.float32)
    got, kernel = run(family, left, right, prec)
    assert kernel == f"mfma_rights_kernel<{prec}>"
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(got, oracle_family(family, l64, r64), oracle_family(family, l64, r64, absval=True))
    assert err <= 2e-6, (family, rows, cols, err)


@pytest.mark.parametrize("prec,side,value", [("bf16x3", "left", np.inf), ("bf16x3", "right", np.nan),
                                             ("fp16x3", "right", 1e5), ("bf16x3", "left", 3.4e38)])
def test_values_that_the_split_does_not_hold(prec, side, value):
    """Such a batch gets the results of the default tile, and the next one is unaffected."""
    left = seeded((2, 50, 40), "u11", 73, np.float32)
    right = seeded((60, 50, 40), "u11", 74, np.float32)
    clean, kernel = run("n_to_m", left, right, prec)
    assert kernel == f"mfma_rights_kernel<{prec}>"
    l, r = left.copy(), right.copy()
    if side == "left":
        l[1, 49, 39] = value
    else:
        r[59, 0, 0] = value
    got, _ = run("n_to_m", l, r, prec)
    tiles, kernel = run("n_to_m", l, r, prec, tile=6)
    assert kernel == f"mfma_kernel<{prec}>"
    np.testing.assert_array_equal(got, tiles)
    again, _ = run("n_to_m", left, right, prec)
    np.testing.assert_array_equal(again, clean)


@pytest.mark.parametrize("prec,value", [("bf16x3", np.nan), ("fp16x3", 1e5)])
def test_values_that_the_split_does_not_hold_above_64_columns(prec, value):
    """The same where the default tile is the one of rows kernels."""
    left = seeded((1, 50, 81), "u11", 75, np.float32)
    right = seeded((50, 50, 81), "u11", 76, np.float32)
    clean, kernel = run("one_to_many", left, right, prec)
    assert kernel == f"mfma_rights_kernel<{prec}>"
    r = right.copy()
    r[49, 7, 80] = value
    got, _ = run("one_to_many", left, r, prec)
    tiles, kernel = run("one_to_many", left, r, prec, tile=9)
    assert kernel == f"mfma_rows_kernel<{prec}>"
    np.testing.assert_array_equal(got, tiles)
    again, _ = run("one_to_many", left, right, prec)
    np.testing.assert_array_equal(again, clean)
