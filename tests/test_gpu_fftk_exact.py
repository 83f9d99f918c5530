"""GPU accuracy of the own FFT on double data.  Inputs are whole numbers of up to 1000, so that the
definition's sums are exact in float64, and the error in the 2-norm is the transforms' own: a few units
of 2^-53, which powers and rotations of the twiddles' roots had made up to 1.8 times larger.  Bars: what
the same transforms give with a short radix first and powers formed one by one, 1.15 times."""
import numpy as np
import pytest

from xc_testutil import oracle_family, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# rows, cols, relative error in the 2-norm of unsigned and of signed data
SIZES = [(16, 16, 2.69e-16, 5.28e-16), (64, 64, 2.27e-16, 5.84e-16), (64, 32, 2.58e-16, 5.77e-16),
         (90, 90, 3.12e-16, 6.31e-16), (100, 120, 3.20e-16, 6.83e-16), (130, 130, 3.06e-16, 5.97e-16),
         (180, 100, 3.26e-16, 6.68e-16), (20, 257, 2.90e-16, 5.90e-16), (300, 60, 2.95e-16, 6.31e-16),
         (12, 1000, 3.01e-16, 7.22e-16), (1000, 12, 3.41e-16, 6.70e-16)]


@pytest.mark.parametrize("signed", [False, True])
@pytest.mark.parametrize("rows,cols,unsigned_err,signed_err", SIZES)
def test_error_in_the_2_norm(rows, cols, unsigned_err, signed_err, signed):
    x = xcorr()
    wrong = total = 0.0
    for seed in range(3):
        rng = np.random.default_rng(700 + seed)
        left, right = (rng.integers(-1000 * signed, 1001, (k, rows, cols)).astype(np.float64) for k in (1, 3))
        out = x.cross_corr("one_to_many", torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda(),
                           precision="fft64", tile=1).cpu().numpy()
        ref = oracle_family("one_to_many", left, right)
        wrong += ((out.reshape(ref.shape) - ref) ** 2).sum()
        total += (ref ** 2).sum()
    err = (wrong / total) ** 0.5
    print(rows, cols, signed, err)
    assert err <= 1.15 * (signed_err if signed else unsigned_err)
