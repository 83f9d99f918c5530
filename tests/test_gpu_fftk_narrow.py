"""GPU parity of the own FFT where its rows have 48 and 96 points, whose blocks write several output rows
at once (widths at both ends of these lengths, heights that end inside a block), and of flat matrices on
both sides of the line between the one-block kernels and rows of 384 points; float and double data."""
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


@pytest.mark.parametrize("dtype,tol", [(np.float32, 1e-6), (np.float64, 1e-9)])
@pytest.mark.parametrize("rows,cols,small", [(1, 128, True), (1, 129, False), (16, 129, False), (9, 192, False),
                                             (2, 193, True), (16, 193, True), (17, 150, False)]
                         + [(8, 64, True), (8, 65, False), (1, 96, False), (9, 65, True), (8, 97, True)])
def test_flat(rows, cols, small, dtype, tol):
    left, right = seeded((2, rows, cols), "u11", 63, dtype), seeded((3, rows, cols), "u01", 64, dtype)
    x = xcorr()
    out = torch.full(x.result_shape("n_to_m", rows, cols, 2, 3), float("nan"), device="cuda",
                     dtype=torch.from_numpy(left).dtype)
    x.cross_corr("n_to_m", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fft64",
                 tile=1)
    torch.cuda.synchronize()
    assert (x.last_launch()["kernel"] == "fftk_small_pairs") == small
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(out.cpu().numpy(), oracle_family("n_to_m", l64, r64),
                        oracle_family("n_to_m", l64, r64, absval=True))
    assert err <= tol, (rows, cols, err)


def test_flat_batch():
    """One plan over both sides of the line, in one class each."""
    x = xcorr()
    sizes = [(1, 129), (16, 192), (10, 193), (16, 256), (5, 150), (12, 130), (17, 150), (3, 384), (20, 200)]
    left = seeded((1, sum(r * c for r, c in sizes)), "u11", 65, np.float32)[0]
    right = seeded((1, left.size), "u01", 66, np.float32)[0]
    pairs, off, oo = [], 0, 0
    for r, c in sizes:
        pairs.append((off, off, oo, r, c))
        off += r * c
        oo += (2 * r - 1) * (2 * c - 1)
    plan = x.BatchPlan(pairs, "fft64", tile=1)
    out = torch.full((oo,), float("nan"), device="cuda")
    plan.run(torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    plan.close()
    for lo, ro, o, r, c in pairs:
        lm, rm = (a[lo:lo + r * c].reshape(1, r, c).astype(np.float64) for a in (left, right))
        res = got[o:o + (2 * r - 1) * (2 * c - 1)].reshape(1, 2 * r - 1, 2 * c - 1)
        err, _ = norm_error(res, oracle_family(0, lm, rm), oracle_family(0, lm, rm, absval=True))
        assert err <= 1e-6, (r, c, err)
