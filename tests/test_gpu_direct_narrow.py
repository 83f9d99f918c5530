"""GPU checks of the FP32 direct method's default kernel for batches of narrow matrices, and of single
rows, with many rights per left: the kernel taken on either side of each line, and parity with the CPU
oracle (normalised error <= 1e-6)."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

PAIRS, MATRIX = "direct_pairs_kernel<f32> ty4 tx4", "direct_pairs_kernel<f32> matrix instructions"


@pytest.mark.parametrize("family,rows,cols,n,m,kernel", [
    ("n_to_m", 142, 1, 20, 186, PAIRS), ("n_to_m", 90, 4, 12, 110, PAIRS), ("n_to_mn", 178, 3, 22, 1320, PAIRS),
    ("n_to_m", 66, 5, 8, 272, PAIRS), ("n_to_m", 62, 7, 20, 120, PAIRS), ("n_to_m", 60, 12, 29, 64, PAIRS),
    ("n_to_m", 60, 13, 29, 64, MATRIX), ("n_to_m", 100, 15, 4, 100, MATRIX),
    ("one_to_many", 1, 87, 1, 12316, PAIRS), ("one_to_many", 1, 40, 1, 12316, MATRIX),
    ("n_to_mn", 1, 41, 3, 27000, PAIRS)])
def test_kernel_and_parity(family, rows, cols, n, m, kernel):
    x = xcorr()
    left, right = seeded((n, rows, cols), "u01", 81, np.float32), seeded((m, rows, cols), "u11", 82, np.float32)
    out = torch.full(x.result_shape(family, rows, cols, n, m), float("nan"), device="cuda")
    print(f"narrow {family} {left.shape} {right.shape}", flush=True)
    x.cross_corr(family, torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(), out=out, precision="fp32")
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"] == kernel
    l64, r64 = left.astype(np.float64), right.astype(np.float64)
    err, _ = norm_error(out.cpu().numpy(), oracle_family(family, l64, r64), oracle_family(family, l64, r64, absval=True))
    assert err <= 1e-6, (family, rows, cols, err)
