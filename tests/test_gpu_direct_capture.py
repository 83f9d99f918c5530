"""GPU checks of the direct method's default kernel inside a graph captured on a stream without a
workspace: the call takes a kernel that needs none."""
import numpy as np
import pytest

from xc_testutil import norm_error, oracle_family, seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype,bar", [(np.float32, 1e-6), (np.float64, 1e-12)])
def test_many_rights_without_a_workspace(dtype, bar):
    """64 rights of 128x100, which the kernels with copied inputs serve otherwise."""
    x = xcorr()
    left, right = seeded((1, 128, 100), "u01", 81, dtype), seeded((64, 128, 100), "u11", 82, dtype)
    l, r = torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda()
    x.cross_corr("one_to_many", l, r, precision="fp32")
    assert x.last_launch()["kernel"].startswith("direct_pairs_kernel")
    out = torch.empty((64, 255, 199), dtype=l.dtype, device="cuda")
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        x.cross_corr("one_to_many", l, r, out=out, precision="fp32")
    assert x.last_launch()["kernel"].startswith("direct_kernel")
    l64, r64 = left.astype(np.float64), right[[0, 63]].astype(np.float64)
    ref, scale = oracle_family("one_to_many", l64, r64), oracle_family("one_to_many", l64, r64, absval=True)
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.isfinite(got).all()
        assert norm_error(got[[0, 63]], ref, scale)[0] <= bar
        _ = (out * 2).sum().item()
