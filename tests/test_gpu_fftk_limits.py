"""GPU checks of the own FFT's one-block kernels at the limits of a call: more pairs than one launch
holds threads for, and batches whose padded spectra would take many times the memory of the
three-pass layout."""
import numpy as np
import pytest

from xc_testutil import seeded, xcorr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_more_pairs_than_one_launch_holds():
    """8192 x 8193 pairs of 1x1: 64 threads each are more than 2^32.  A result is one product."""
    x = xcorr()
    left = seeded((8192, 1, 1), "normal", 1, np.float32)
    right = seeded((8193, 1, 1), "normal", 2, np.float32)
    dl, dr = torch.from_numpy(left).cuda(), torch.from_numpy(right).cuda()
    out = torch.full((8192 * 8193, 1, 1), float("nan"), device="cuda")
    print("8192 x 8193 of 1x1", flush=True)
    x.cross_corr("n_to_m", dl, dr, out=out, precision="fft64", tile=1)
    torch.cuda.synchronize()
    assert x.last_launch()["kernel"] == "fftk_small_pairs"
    got = out.view(8192, 8193).double()
    ref = dl.view(-1, 1).double() * dr.view(1, -1).double()
    assert ((got - ref).abs() <= 1e-6 * ref.abs()).all()


def grown_by(call):
    """Device memory taken by `call`, in bytes."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    call()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


def flat_rights(m):
    """One left and m rights of 1x256, whose padded spectra are 32 times the three-pass layout's."""
    left = torch.from_numpy(seeded((1, 1, 256), "normal", 3, np.float32)).cuda()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    return left, torch.randn((m, 1, 256), generator=gen, device="cuda"), torch.full((m, 1, 511), float("nan"), device="cuda")


def check_rows(left, right, out):
    """Every 101st result against float64, and every one written."""
    assert not out.isnan().any()
    wide = torch.nn.functional.pad(left[0, 0].double(), (255, 255)).unfold(0, 256, 1)
    r64 = right[::101, 0].double()
    err = (out[::101, 0].double() - r64 @ wide.T).abs() / (r64.abs() @ wide.abs().T)
    assert err.max().item() <= 1e-6  # the own FFT's bar


def test_many_flat_rights_in_one_call():
    """300 000 rights: 1.2 GB of row spectra and 2 GiB of Z, where padded spectra take 39 GB."""
    x = xcorr()
    left, right, out = flat_rights(300_000)
    with torch.cuda.stream(torch.cuda.Stream()):  # workspaces of its own
        torch.cuda.synchronize()
        print("1 x 300000 of 1x256", flush=True)
        grown = grown_by(lambda: x.cross_corr("one_to_many", left, right, out=out, precision="fft64", tile=1))
    assert grown <= 8 << 30
    check_rows(left, right, out)


def test_many_flat_rights_in_one_plan():
    """40 000 pairs: 0.5 GB of S and Z, where padded spectra take 5.3 GB; with and without the graph."""
    x = xcorr()
    left, right, out = flat_rights(40_000)
    pairs = [(0, 256 * i, 511 * i, 1, 256) for i in range(40_000)]
    plans = []
    grown = grown_by(lambda: plans.append(x.BatchPlan(pairs, "fft64", tile=1, branches=4)))
    assert grown <= 2 << 30
    for graph in (False, True, True):
        out.fill_(float("nan"))
        plans[0].run(left, right, out, use_graph=graph)
        torch.cuda.synchronize()
        check_rows(left, right, out)
    plans[0].close()
