"""GPU parity of the own FFT's one-block kernels (padded lengths 2^a x 2^b of at most 16384
values, each 32..512) against the CPU oracle, at the edges of their lengths.

Bars (normalised error = |x - x64| / corr(|L|,|R|)): float data 1e-6 (FP64 transforms, FP32
results), double data 1e-9, as for the other own-FFT kernels: the transform's rounding, about
1e-16 of the sum of all products, over a single product at the one-element-overlap corners.
"""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# rows, cols, taken by the one-block kernels
SIZES = [(1, 1, True), (1, 256, True), (256, 1, True), (16, 16, True), (17, 16, True), (16, 17, True), (32, 33, True),
         (33, 32, True), (64, 64, True), (63, 61, True), (128, 32, True), (32, 128, True), (16, 256, True),
         (256, 16, True), (64, 65, False), (65, 64, False), (17, 256, False), (257, 3, False), (3, 257, False)]
FAMILIES = [("one_to_one", 1, 1), ("one_to_many", 1, 5), ("n_to_mn", 3, 6), ("n_to_m", 3, 5)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows,cols,small", SIZES)
def test_edges(rows, cols, small, dtype):
    x = xcorr()
    for k, (family, n, m) in enumerate(FAMILIES if rows * cols <= 4096 else FAMILIES[2:3]):
        print(f"{family} {rows}x{cols} {dtype.__name__}", flush=True)
        left = seeded((n, rows, cols), "normal", 70 + k, dtype)
        right = seeded((m, rows, cols), "u11", 80 + k, dtype)
        shape = x.result_shape(family, rows, cols, n, m)
        out = torch.full(shape, float("nan"), device="cuda", dtype=torch.from_numpy(left).dtype)
        x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out,
                     precision="fft64", tile=1 + k % 2)
        torch.cuda.synchronize()
        assert (x.last_launch()["kernel"] == "fftk_small_pairs") == small
        l64, r64 = left.astype(np.float64), right.astype(np.float64)
        ref = oracle_family(family, l64, r64)
        err, _ = norm_error(out.cpu().numpy(), ref, oracle_family(family, l64, r64, absval=True))
        assert err <= (1e-6 if dtype is np.float32 else 1e-9), (family, rows, cols, err)


def test_uneven_batch_of_small_matrices():
    """One plan over sizes from 1 to 64 (several of them in one class, smaller than its lengths),
    with and without the graph."""
    x = xcorr()
    sizes = [(1, 1), (2, 7), (16, 16), (16, 17), (20, 9), (31, 64), (33, 33), (64, 64), (60, 41), (5, 130)]
    left = seeded((1, sum(r * c for r, c in sizes)), "u11", 91, np.float32)[0]
    right = seeded((1, left.size), "normal", 92, np.float32)[0]
    pairs, off, oo = [], 0, 0
    for r, c in sizes:
        pairs.append((off, off, oo, r, c))
        off += r * c
        oo += (2 * r - 1) * (2 * c - 1)
    plan = x.BatchPlan(pairs, "fft64", tile=1, branches=2)
    dl, dr = torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda()
    for graph in (False, True, True):
        out = torch.full((oo,), float("nan"), device="cuda")
        plan.run(dl, dr, out, use_graph=graph)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        for lo, ro, o, r, c in pairs:
            lm = left[lo:lo + r * c].reshape(1, r, c).astype(np.float64)
            rm = right[ro:ro + r * c].reshape(1, r, c).astype(np.float64)
            res = got[o:o + (2 * r - 1) * (2 * c - 1)].reshape(1, 2 * r - 1, 2 * c - 1)
            err, _ = norm_error(res, oracle_family(0, lm, rm), oracle_family(0, lm, rm, absval=True))
            assert err <= 1e-6, (r, c, err)
    plan.close()


# rows, cols, lefts, rights: more pairs than the chip holds with one column per thread
MANY = [(64, 64, 5, 52), (16, 200, 5, 52), (200, 16, 5, 52), (30, 100, 5, 52), (100, 30, 5, 52), (60, 30, 9, 58),
        (30, 60, 9, 58), (120, 16, 9, 58), (16, 120, 9, 58), (30, 30, 19, 54), (16, 60, 19, 54), (60, 16, 19, 54),
        (16, 30, 33, 63), (30, 16, 33, 63)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows,cols,n,m", MANY)
def test_many_pairs(rows, cols, n, m, dtype):
    """Two columns per thread: the first and last matrices against the oracle, every pair against the
    one-left calls (one column per thread).  Those differ by the transforms' rounding, below 1e-14
    of the norms' product, and one rounding of the output."""
    x = xcorr()
    left = seeded((n, rows, cols), "normal", 95, dtype)
    right = seeded((m, rows, cols), "u11", 96, dtype)
    dl, dr = torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda()
    out = x.cross_corr("n_to_m", dl, dr, precision="fft64", tile=1)
    threads = x.last_launch()["block"]
    got = out.cpu().numpy().reshape(n, m, 2 * rows - 1, 2 * cols - 1)
    parts = [x.cross_corr("one_to_many", dl[k:k + 1], dr, precision="fft64", tile=1) for k in range(n)]
    assert x.last_launch()["block"] != threads
    one = torch.stack(parts).cpu().numpy().reshape(got.shape).astype(np.float64)
    norm = np.sqrt((left.astype(np.float64) ** 2).sum((1, 2))[:, None] * (right.astype(np.float64) ** 2).sum((1, 2)))
    bound = 1e-14 * norm[:, :, None, None] + np.finfo(dtype).eps * np.abs(one)
    assert (np.abs(got - one) <= bound).all()
    l64, r64 = left[[0, -1]].astype(np.float64), right[[0, -1]].astype(np.float64)
    ref = oracle_family("n_to_m", l64, r64)
    err, _ = norm_error(got[np.ix_([0, n - 1], [0, m - 1])].reshape(ref.shape), ref,
                        oracle_family("n_to_m", l64, r64, absval=True))
    assert err <= (1e-6 if dtype is np.float32 else 1e-9), (rows, cols, err)
