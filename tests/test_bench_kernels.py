"""bench.py's accounts of the library's kernels: a kernel whose bytes it does not know is priced as
matrix-core arithmetic."""
import importlib.util
import pathlib
import re

import pytest

REPO = pathlib.Path(__file__).resolve().parent.parent


def bench():
    spec = importlib.util.spec_from_file_location("bench_under_test", REPO / "bench.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def fft_timers():
    """Names of the FFT methods' kernel timers, from the sources."""
    names = set()
    for path in sorted((REPO / "cross-corr_amd" / "csrc").glob("xc_fft*.hip")):
        names |= set(re.findall(r'(?:launch_timed|timed \w+)\("(\w+)"', path.read_text()))
    return sorted(names)


def test_every_fft_kernel_has_its_bytes():
    b = bench()
    names = fft_timers()
    assert {"fftk_rows_fwd", "fftk_small_spec", "fftk_small_pairs", "fft_hadamard"} <= set(names)
    unknown = [n for n in names if b.kernel_bytes(n, 64, 64, 16, 64, 1024) is None]
    assert unknown == []


@pytest.mark.parametrize("rows,cols,lr,lc", [(64, 64, 128, 128), (10, 10, 32, 32), (60, 30, 128, 64)])
def test_one_block_kernels(rows, cols, lr, lc):
    b = bench()
    half = lr * (lc // 2 + 1) * 16
    assert b.kernel_bytes("fftk_small_spec", rows, cols, 2, 3, 6) == 5 * (rows * cols * 4 + half)
    assert (b.kernel_bytes("fftk_small_pairs", rows, cols, 2, 3, 6)
            == 5 * half + 6 * (2 * rows - 1) * (2 * cols - 1) * 4)
    out = 6 * (2 * rows - 1) * (2 * cols - 1)
    assert b.kernel_bytes("fftk_small_pairs", rows, cols, 2, 3, 6, elem=8) == 5 * half + out * 8
