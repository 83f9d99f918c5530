"""GPU parity of the FP32 direct method on the FP32 matrix instructions (the default for batches with
many rights per left) against the CPU oracle: partial groups of 16 rights, tiles of 4 dy x 16 dx that
cross the result's edges, steps of 16 columns that cross the matrix's, fewer steps than waves, every
family; data that is not finite; a call under graph capture.  Bar of the FP32 direct method:
normalised error <= 1e-6 (products summed in FP32 partials of 32, added in FP64)."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NAME = "direct_pairs_kernel<f32> matrix instructions"


def run(family, left, right, **kw):
    x = xcorr()
    shape = x.result_shape(family, left.shape[1], left.shape[2], left.shape[0], right.shape[0])
    out = torch.full(shape, float("nan"), device="cuda")
    print(f"matrix {family} {left.shape} {right.shape}", flush=True)
    x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fp32", **kw)
    torch.cuda.synchronize()
    return out.cpu().numpy(), x.last_launch()["kernel"]


@pytest.mark.parametrize("dist", ["u01", "normal"])
@pytest.mark.parametrize("family,rows,cols,n,m", [
    ("n_to_mn", 33, 47, 4, 128), ("one_to_many", 20, 200, 1, 100), ("one_to_many", 500, 3, 1, 160),
    ("one_to_many", 64, 63, 1, 65), ("n_to_m", 50, 41, 20, 17), ("one_to_many", 32, 32, 1, 256),
    ("one_to_many", 1, 2000, 1, 64), ("n_to_mn", 60, 49, 5, 65), ("one_to_many", 66, 65, 1, 48),
    ("n_to_m", 31, 16, 40, 31), ("n_to_m", 17, 17, 40, 48)])
def test_parity(family, rows, cols, n, m, dist):
    left = seeded((n, rows, cols), dist, 61, np.float32)
    right = seeded((m, rows, cols), dist, 62, np.float32)
    got, kernel = run(family, left, right)
    assert kernel == NAME
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(got, oracle_family(family, l64, r64), oracle_family(family, l64, r64, absval=True))
    assert err <= 1e-6, (family, rows, cols, err)


@pytest.mark.parametrize("side,value", [("left", np.inf), ("right", np.nan), ("right", -np.inf)])
def test_values_that_are_not_finite(side, value):
    """Such a batch gets the results of the lanes-over-pairs kernel, and the next one is unaffected."""
    left = seeded((2, 50, 40), "u11", 63, np.float32)
    right = seeded((40, 50, 40), "u11", 64, np.float32)
    clean, kernel = run("n_to_m", left, right)
    assert kernel == NAME
    l, r = left.copy(), right.copy()
    if side == "left":
        l[1, 49, 39] = value
    else:
        r[39, 0, 0] = value
    got, _ = run("n_to_m", l, r)
    pairs, kernel = run("n_to_m", l, r, tile=2)
    assert kernel.startswith("direct_pairs_kernel<f32> ty4")
    assert not np.isfinite(got).all()
    np.testing.assert_array_equal(got, pairs)
    again, _ = run("n_to_m", left, right)
    np.testing.assert_array_equal(again, clean)


def test_capture_without_a_workspace_takes_the_kernel_that_needs_none():
    x = xcorr()
    left, right = seeded((1, 96, 80), "u01", 65, np.float32), seeded((32, 96, 80), "u01", 66, np.float32)
    eager, kernel = run("one_to_many", left, right)
    assert kernel == NAME
    l, r = torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda()
    out = torch.empty(eager.shape, device="cuda")
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        x.cross_corr("one_to_many", l, r, out=out, precision="fp32")
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_allclose(out.cpu().numpy(), eager, rtol=2e-6)  # positive data: the bar, twice
        _ = (out * 2).sum().item()
