"""GPU checks of the FP32 direct method's default kernel for one right per left, where the 16 x 16 shifts
and the register tiles take turns: the kernel taken at shapes measured well to either side of the
line, and parity with the CPU oracle (normalised error <= 1e-6)."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TILES, SHIFTS = "direct_kernel<f32> ty", "direct_kernel<f32> 16x16 shifts"


@pytest.mark.parametrize("family,rows,cols,n,m,kernel", [
    ("one_to_one", 129, 37, 1, 1, TILES), ("one_to_one", 26, 335, 1, 1, TILES), ("one_to_one", 65, 124, 1, 1, TILES),
    ("one_to_one", 64, 128, 1, 1, TILES),
    ("n_to_mn", 13, 146, 3, 3, TILES), ("one_to_many", 8, 76, 1, 1, TILES), ("one_to_one", 54, 61, 1, 1, SHIFTS),
    ("one_to_one", 130, 130, 1, 1, SHIFTS), ("one_to_one", 256, 64, 1, 1, SHIFTS),
    ("one_to_one", 17, 17, 1, 1, SHIFTS), ("n_to_mn", 34, 72, 2, 2, SHIFTS),
    ("one_to_many", 129, 37, 1, 2, SHIFTS)])
def test_kernel_and_parity(family, rows, cols, n, m, kernel):
    x = xcorr()
    left, right = seeded((n, rows, cols), "u01", 95, np.float32), seeded((m, rows, cols), "u11", 96, np.float32)
    out = torch.full(x.result_shape(family, rows, cols, n, m), float("nan"), device="cuda")
    print(f"single {family} {left.shape} {right.shape}", flush=True)
    x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fp32")
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"].startswith(kernel)
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(out.cpu().numpy(), oracle_family(family, l64, r64), oracle_family(family, l64, r64, absval=True))
    assert err <= 1e-6, (family, rows, cols, err)


@pytest.mark.parametrize("rows,cols,m", [(100, 12, 6), (16, 16, 4), (60, 16, 3), (130, 9, 5)])
@pytest.mark.parametrize("dist", ["u01", "u11", "normal"])
def test_narrow_matrices_are_as_exact_as_by_the_register_tiles(rows, cols, m, dist):
    """Relative error in the 2-norm over several batches, against the kernel that served them before."""
    x = xcorr()
    wrong, total = {0: 0.0, 1: 0.0}, 0.0
    for seed in range(8):
        left, right = seeded((1, rows, cols), dist, 300 + seed, np.float32), seeded((m, rows, cols), dist, 400 + seed, np.float32)
        ref = oracle_family("one_to_many", left.astype(np.float64), right.astype(np.float64))
        total += (ref ** 2).sum()
        for tile in wrong:
            out = x.cross_corr("one_to_many", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(),
                               precision="fp32", tile=tile)
            assert x.last_launch()["kernel"].startswith(TILES if tile else SHIFTS)
            wrong[tile] += ((out.cpu().numpy().astype(np.float64).reshape(ref.shape) - ref) ** 2).sum()
    print(rows, cols, dist, [(v / total) ** 0.5 for v in wrong.values()])
    assert wrong[0] <= wrong[1]
