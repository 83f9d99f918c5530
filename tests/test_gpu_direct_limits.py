"""GPU checks of the FP32 direct method where a kernel's grid would be 2^32 threads or more (the grid
size wraps there, without an error): the call takes a kernel whose grid fits."""
import numpy as np
import pytest

from xc_testutil import seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("cols,n,m", [(1, 20_000_000, 4),    # 16 x 16 shifts: 80 M tiles of 64 threads
                                      (16, 8_400_000, 12)])  # matrix kernel: 16.8 M blocks of 256 threads
def test_more_tiles_than_one_launch_holds(cols, n, m):
    """n_to_m of 1 x cols: every result written, every 997th left's results against float64."""
    x = xcorr()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    left = torch.rand((n, 1, cols), generator=gen, device="cuda")
    right = torch.rand((m, 1, cols), generator=gen, device="cuda")
    out = torch.full((n * m, 1, 2 * cols - 1), float("nan"), device="cuda")
    print(f"{n} x {m} of 1x{cols}", flush=True)
    x.cross_corr("n_to_m", left, right, out=out, precision="fp32")
    torch.cuda.synchronize()
    got = out.view(n, m, 2 * cols - 1)
    for part in got.split(1 << 20):
        assert not part.isnan().any()
    # out[dx + cols - 1] = sum_c left[c + dx] right[c]; positive data: the bar is relative
    l64 = left[::997, 0].double().cpu()
    wide = torch.nn.functional.pad(l64, (cols - 1, cols - 1)).unfold(1, cols, 1)
    ref = torch.tensordot(wide, right[:, 0].double().cpu(), dims=([2], [1])).transpose(1, 2)
    np.testing.assert_allclose(got[::997].cpu().numpy(), ref.numpy(), rtol=1e-6)


def test_copies_of_many_lefts_are_bounded():
    """15 M lefts of 1x1, 60 MB: padded for the matrix kernel they would take 23 GB."""
    x = xcorr()
    n, m = 15_000_000, 8
    left = torch.rand((n, 1, 1), device="cuda")
    right = torch.rand((m, 1, 1), device="cuda")
    out = torch.full((n * m, 1, 1), float("nan"), device="cuda")
    with torch.cuda.stream(torch.cuda.Stream()):  # a workspace of its own
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        print(f"{n} x {m} of 1x1", flush=True)
        x.cross_corr("n_to_m", left, right, out=out, precision="fp32")
        torch.cuda.synchronize()
        assert before - torch.cuda.mem_get_info()[0] <= 16 << 30
    ref = left.view(n, 1) * right.view(1, m)  # one product each, rounded once
    assert torch.equal(out.view(n, m), ref)
