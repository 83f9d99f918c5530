"""GPU parity of the own FFT's column kernels against the CPU oracle where few pairs share a left
matrix or few waves are in flight: one block transforms the left columns itself and keeps them
over one or two consecutive pairs, which may belong to different lefts.

Bars (normalised error = |x - x64| / corr(|L|,|R|)): float data 1e-6, double data 1e-9, as for the
other own-FFT kernels.
"""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# One column length each; the first of a length has one pair per block (few waves), the second
# two, with an odd number of pairs per left so that blocks cross from one left to the next.
CASES = [("one_to_one", 70, 66, 1, 1), ("n_to_m", 66, 70, 2, 3),      # 256 points
         ("n_to_mn", 7, 300, 4, 12), ("n_to_mn", 7, 300, 121, 363),   # 16 points, 32 columns per wave
         ("n_to_mn", 129, 129, 3, 9), ("n_to_mn", 129, 129, 9, 27),   # 512 points
         ("one_to_many", 257, 20, 1, 5), ("n_to_mn", 257, 20, 25, 75),  # 1024 points, two waves per column
         ("n_to_mn", 520, 10, 2, 6)]                                  # 2048 points


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("family,rows,cols,n,m", CASES)
def test_grouped_columns(family, rows, cols, n, m, dtype):
    x = xcorr()
    left = seeded((n, rows, cols), "normal", 51, dtype)
    right = seeded((m, rows, cols), "u11", 52, dtype)
    out = x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), precision="fft64",
                       tile=1).cpu().numpy()
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    ref = oracle_family(family, l64, r64)
    err, _ = norm_error(out.reshape(ref.shape), ref, oracle_family(family, l64, r64, absval=True))
    assert err <= (1e-6 if dtype is np.float32 else 1e-9), (family, rows, cols, err)


def test_batch_with_shared_and_alternating_lefts():
    """Pairs of one class whose lefts alternate, repeat and differ in size, with and without the graph."""
    x = xcorr()
    sizes = [(129, 129), (140, 135), (150, 150), (131, 180)]
    left = seeded((1, sum(r * c for r, c in sizes)), "u11", 53, np.float32)[0]
    right = seeded((1, 8 * left.size), "normal", 54, np.float32)[0]
    starts = np.cumsum([0] + [r * c for r, c in sizes])
    pairs, ro, oo = [], 0, 0
    for s in (0, 1, 0, 0, 2, 1, 1, 1, 3, 3, 0, 2, 2, 1, 3, 2, 0):
        r, c = sizes[s]
        pairs.append((int(starts[s]), ro, oo, r, c))
        ro += r * c
        oo += (2 * r - 1) * (2 * c - 1)
    plan = x.BatchPlan(pairs, "fft64", tile=1, branches=2)
    dl, dr = torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda()
    for graph in (False, True, True):
        out = torch.full((oo,), float("nan"), device="cuda")
        plan.run(dl, dr, out, use_graph=graph)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        for lo, r0, o0, r, c in pairs:
            l64 = left[lo:lo + r * c].reshape(1, r, c).astype(np.float64)
            r64 = right[r0:r0 + r * c].reshape(1, r, c).astype(np.float64)
            ref = oracle_family("one_to_one", l64, r64)
            err, _ = norm_error(got[o0:o0 + ref.size].reshape(ref.shape), ref,
                                oracle_family("one_to_one", l64, r64, absval=True))
            assert err <= 1e-6, (r, c, err)
