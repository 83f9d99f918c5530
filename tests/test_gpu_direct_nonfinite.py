"""GPU checks of the FP32 direct method's 16 x 16 shifts kernel on data with infinities and NaNs: a
shift shows one exactly where the sum over its overlap does (CPU oracle), and the sums of all other
shifts are those of the same data with finite values in these places, bit for bit."""
import numpy as np
import pytest

from xc_testutil import oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def run(family, left, right):
    x = xcorr()
    shape = x.result_shape(family, left.shape[1], left.shape[2], left.shape[0], right.shape[0])
    out = torch.full(shape, 7.0, device="cuda")
    print(f"shifts {family} {left.shape} {right.shape}", flush=True)
    x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fp32")
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"].startswith("direct_kernel<f32> 16x16 shifts")
    return out.cpu().numpy()


def spoil(a, kind, rng):
    values = {"nan": [np.nan], "inf": [np.inf], "mixed": [np.nan, np.inf, -np.inf]}[kind.split()[-1]]
    if kind.startswith("half"):
        a[:, :, : a.shape[2] // 2] = values[0]
        return
    for k in range(a.shape[0]):
        for v in values:
            a[k, rng.integers(a.shape[1]), rng.integers(a.shape[2])] = v
    a[0, 0, 0] = values[0]
    a[-1, -1, -1] = values[-1]


@pytest.mark.parametrize("kind", ["nan", "inf", "mixed", "half nan", "half inf"])
@pytest.mark.parametrize("side", ["left", "right", "both"])
@pytest.mark.parametrize("family,rows,cols,n,m", [
    ("one_to_many", 10, 10, 1, 3),   # one panel, groups of two or three rows
    ("one_to_many", 3, 40, 1, 2),    # fewer rows than groups
    ("n_to_m", 33, 47, 2, 2),        # columns and rows that end inside a panel
    ("one_to_many", 70, 100, 1, 3),  # several panels each way
    ("n_to_mn", 101, 20, 2, 2)])
def test_only_the_overlaps_show_it(family, rows, cols, n, m, side, kind):
    rng = np.random.default_rng(5)
    left, right = seeded((n, rows, cols), "u01", 91, np.float32), seeded((m, rows, cols), "u01", 92, np.float32)
    right[:, :, 7 % cols] = 0.0  # an infinity times 0 inside an overlap is NaN
    clean = run(family, left, right)
    l, r = left.copy(), right.copy()
    if side != "right":
        spoil(l, kind, rng)
    if side != "left":
        spoil(r, kind, rng)
    got = run(family, l, r)
    with np.errstate(invalid="ignore"):
        ref = oracle_family(family, l.astype(np.float64), r.astype(np.float64))
    fine = np.isfinite(ref)
    assert (~fine).any()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    shown = ~fine & ~np.isnan(ref)
    np.testing.assert_array_equal(got[shown], ref[shown].astype(np.float32))
    np.testing.assert_array_equal(got[fine], clean[fine])


@pytest.mark.parametrize("kind", ["nan", "mixed"])
@pytest.mark.parametrize("family,rows,cols,n,m", [("one_to_many", 90, 80, 1, 16), ("n_to_m", 33, 47, 12, 20),
                                                  ("n_to_mn", 64, 50, 3, 48), ("one_to_many", 128, 300, 1, 9)])
def test_behind_the_matrix_kernel(family, rows, cols, n, m, kind):
    """Up to 39 rights per left the matrix kernel leaves such a batch to the register tiles, and serves
    finite data after it as before."""
    x = xcorr()
    rng = np.random.default_rng(6)
    left, right = seeded((n, rows, cols), "u01", 93, np.float32), seeded((m, rows, cols), "u01", 94, np.float32)
    shape = x.result_shape(family, rows, cols, n, m)

    def call(l, r, kernel="direct_pairs_kernel<f32> matrix instructions", **kw):
        out = torch.full(shape, 7.0, device="cuda")
        print(f"matrix {family} {l.shape} {r.shape}", flush=True)
        x.cross_corr(family, torch.from_numpy(l).cuda(), torch.from_numpy(r).cuda(), out=out, precision="fp32", **kw)
        torch.cuda.synchronize()
        assert x.last_launch()["kernel"].startswith(kernel)
        return out.cpu().numpy()

    clean = call(left, right)
    r = right.copy()
    spoil(r[m // 2:m // 2 + 1], kind, rng)
    got = call(left, r)
    assert not np.isfinite(got).all()
    np.testing.assert_array_equal(got, call(left, r, "direct_kernel<f32> ty", tile=1, split=1))
    np.testing.assert_array_equal(call(left, right), clean)
