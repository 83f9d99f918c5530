"""GPU checks of the FP32 direct method's default kernel for batches of up to 12 rows, where the register
tiles, the 16 x 16 shifts and the matrix kernel take turns: the kernel taken at shapes measured well to
either side of the lines, and parity with the CPU oracle (normalised error <= 1e-6)."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TILES, SHIFTS = "direct_kernel<f32> ty", "direct_kernel<f32> 16x16 shifts"
MATRIX = "direct_pairs_kernel<f32> matrix instructions"


@pytest.mark.parametrize("family,rows,cols,n,m,kernel", [
    ("n_to_m", 4, 53, 600, 3, TILES), ("n_to_mn", 5, 75, 200, 1000, MATRIX), ("n_to_mn", 1, 44, 21, 210, TILES),
    ("one_to_many", 2, 21, 1, 655, TILES), ("n_to_m", 3, 19, 389, 2, TILES), ("n_to_m", 6, 33, 300, 4, TILES),
    ("n_to_m", 1, 2, 436, 20, TILES), ("one_to_many", 1, 1, 1, 80, SHIFTS), ("n_to_mn", 3, 14, 9, 63, SHIFTS),
    ("n_to_m", 12, 12, 3, 4, SHIFTS), ("one_to_many", 11, 40, 1, 6, SHIFTS), ("n_to_m", 4, 74, 14, 200, MATRIX),
    ("n_to_mn", 10, 97, 1549, 1549, TILES), ("n_to_mn", 2, 22, 4092, 4092, TILES), ("n_to_mn", 3, 47, 62, 62, TILES),
    ("n_to_mn", 12, 12, 5, 5, SHIFTS),
    ("one_to_many", 2, 298, 1, 223, MATRIX), ("n_to_m", 12, 100, 4, 100, MATRIX)])
def test_kernel_and_parity(family, rows, cols, n, m, kernel):
    x = xcorr()
    left, right = seeded((n, rows, cols), "u01", 83, np.float32), seeded((m, rows, cols), "u11", 84, np.float32)
    out = torch.full(x.result_shape(family, rows, cols, n, m), float("nan"), device="cuda")
    print(f"flat {family} {left.shape} {right.shape}", flush=True)
    x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fp32")
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"].startswith(kernel)
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(out.cpu().numpy(), oracle_family(family, l64, r64), oracle_family(family, l64, r64, absval=True))
    assert err <= 1e-6, (family, rows, cols, err)
