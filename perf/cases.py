"""The calls that the performance of this framework is measured on.

Each case is one call of the Python binding with its inputs resident on the GPU, as a program
that correlates batches of images makes it: the four families of the library, square and
ragged sizes from 10x10 to 1024x1024, float and double data, the AUTO method, the methods that
a caller asks for by name (the definition in FP32, the split-precision MFMA kernel, the
reference's FFT pipeline) and an uneven batch through a reusable plan.
"""
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

FFT_METHODS = ("auto", "batch", "fft")


def package():
    """The framework's Python package (its folder name has a hyphen: loaded by path)."""
    name = "cross_corr_amd"
    if name not in sys.modules:
        path = pathlib.Path.cwd() / "cross-corr_amd" / "__init__.py"
        spec = importlib.util.spec_from_file_location(name, path)
        module = importlib.util.module_from_spec(spec)
        sys.modules[name] = module
        spec.loader.exec_module(module)
    return sys.modules[name]


def case_of(name, method, family, n, m, rows, cols, dtype="float32", values="u01"):
    return {"name": name, "method": method, "family": family, "n": n, "m": m, "rows": rows, "cols": cols,
            "dtype": dtype, "values": values}


def listed():
    return [
        # a handful of the smallest templates: what counts is the latency of the call
        case_of("auto_1x4_10x10", "auto", "one_to_many", 1, 4, 10, 10, values="u11"),
        # registration of one pair of images, one call at a time
        case_of("auto_pair_128", "auto", "one_to_one", 1, 1, 128, 128),
        # one template against a batch of images: the benchmark's headline workload
        case_of("auto_1x64_256", "auto", "one_to_many", 1, 64, 256, 256),
        # every filter against every patch
        case_of("auto_16x64_64", "auto", "n_to_m", 16, 64, 64, 64, values="normal"),
        # the same in double precision
        case_of("auto_16x64_64_f64", "auto", "n_to_m", 16, 64, 64, 64, dtype="float64", values="normal"),
        # several references, each against the frames of its own series; ragged image size
        case_of("auto_5x60_150x203", "auto", "n_to_mn", 5, 60, 150, 203, values="normal"),
        # large images, more results than the caches hold
        case_of("auto_1x32_1024", "auto", "one_to_many", 1, 32, 1024, 1024),
        # regions of many sizes (128 groups of one left and four rights, 16 to 505 wide) in one plan
        {"name": "batch_128x4_16to512", "method": "batch", "groups": 128, "per_group": 4, "lo": 16, "hi": 512,
         "sizes_seed": 2024, "values": "u11"},
        # the definition in FP32: the reference's own algorithm, many rights for each left ...
        case_of("fp32_1x64_256", "fp32", "one_to_many", 1, 64, 256, 256),
        # ... and few of them, of a ragged size
        case_of("fp32_2x6_100x120", "fp32", "n_to_m", 2, 6, 100, 120, values="u11"),
        # the definition on the matrix cores at FP32-like accuracy
        case_of("bf16x3_1x64_256", "bf16x3", "one_to_many", 1, 64, 256, 256),
        # the reference's FFT pipeline (fft_* algorithms) in single precision
        case_of("fft_4x16_200", "fft", "n_to_m", 4, 16, 200, 200),
    ]


def log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["auto", "f64", "batch", "fp32", "split", "fft"], [9, 2, 2, 2, 3, 2])[0]
    values = rng.choice(["u01", "u11", "normal"])
    if kind == "batch":
        return {"method": "batch", "groups": log_uniform(rng, 8, 128), "per_group": rng.randint(1, 4), "lo": 16,
                "hi": log_uniform(rng, 64, 512), "sizes_seed": rng.randrange(1 << 30), "values": values}
    # most images are square or nearly so
    hi = {"auto": 1024, "f64": 192, "fp32": 256, "split": 256, "fft": 400}[kind]
    rows = log_uniform(rng, 10, hi)
    cols = rows if rng.random() < 0.4 else min(hi, max(10, int(rows * rng.uniform(0.6, 1.7))))
    # results of one call: as many as the largest listed case of the kind has work for
    area, out = rows * cols, (2 * rows - 1) * (2 * cols - 1)
    most = {"auto": 1.2e8 / out, "f64": min(3e10 / area ** 2, 3e7 / out), "fp32": 2e11 / area ** 2,
            "split": 2e11 / area ** 2, "fft": 3e7 / out}[kind]
    most = int(max(1, min(most, 1024)))
    family = rng.choice(["one_to_one", "one_to_many", "n_to_mn", "n_to_m"])
    if family == "one_to_one":
        n, m = 1, 1
    elif family == "one_to_many":
        n, m = 1, log_uniform(rng, 1, min(most, 256))
    elif family == "n_to_mn":
        n = log_uniform(rng, 1, min(most, 16))
        m = n * log_uniform(rng, 1, max(1, min(most, 256) // n))
    else:
        n = log_uniform(rng, 1, min(most, 16))
        m = log_uniform(rng, 1, max(1, min(most // n, 64)))
    method = {"auto": "auto", "f64": "auto", "fp32": "fp32", "fft": "fft"}.get(kind) or rng.choice(
        ["bf16x3", "bf16x3", "fp16x3"])
    got = case_of("", method, family, n, m, rows, cols, "float64" if kind == "f64" else "float32", values)
    del got["name"]
    return got


def numbers(shape, values, gen, dtype):
    """Pixel values: intensities in [0, 1), signed values in [-1, 1), or normalised data."""
    if values == "normal":
        return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    x = torch.rand(shape, generator=gen, device="cuda", dtype=dtype)
    return x if values == "u01" else 2 * x - 1


def batch_layout(case):
    """(sizes, pairs, left length, right length, output length) of an uneven batch."""
    u = np.random.RandomState(case["sizes_seed"]).rand(case["groups"])
    sizes = [int(round(case["lo"] * (case["hi"] / case["lo"]) ** x)) for x in u]
    pairs, lo, ro, oo = [], 0, 0, 0
    for s in sizes:
        for _ in range(case["per_group"]):
            pairs.append((lo, ro, oo, s, s))
            ro += s * s
            oo += (2 * s - 1) ** 2
        lo += s * s
    return sizes, pairs, lo, ro, oo


def inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["method"] == "batch":
        _, _, nl, nr, _ = batch_layout(case)
        return tuple(numbers((k,), case["values"], gen, torch.float32) for k in (nl, nr))
    dtype = getattr(torch, case["dtype"])
    return tuple(numbers((k, case["rows"], case["cols"]), case["values"], gen, dtype) for k in (case["n"], case["m"]))


def prepare(case, seed):
    x = package()
    left, right = inputs(case, seed)
    if case["method"] == "batch":
        _, pairs, _, _, length = batch_layout(case)
        out = torch.empty(length, device="cuda")
        return {"x": x, "left": left, "right": right, "out": out, "case": case,
                "plan": x.BatchPlan(pairs, precision="fft64", tile=1, branches=4)}
    shape = x.result_shape(case["family"], case["rows"], case["cols"], case["n"], case["m"])
    return {"x": x, "left": left, "right": right, "case": case, "out": torch.empty(shape, dtype=left.dtype, device="cuda")}


def run(state):
    x, case, left, right, out = (state[k] for k in ("x", "case", "left", "right", "out"))
    if case["method"] == "batch":
        return state["plan"].run(left, right, out)
    if case["method"] == "fft":
        return x.fft_cross_corr(case["family"], left, right, out=out)
    return x.cross_corr(case["family"], left, right, out=out, precision=case["method"])


def results_of(case):
    """[(rows, cols, lefts, rights, results)] of every group of equal matrices."""
    if case["method"] == "batch":
        return [(s, s, 1, case["per_group"], case["per_group"]) for s in batch_layout(case)[0]]
    k = case["n"] * case["m"] if case["family"] == "n_to_m" else case["m"]
    return [(case["rows"], case["cols"], case["n"], case["m"], k)]


def work(case):
    nbytes = flops = 0
    for rows, cols, n, m, k in results_of(case):
        out = (2 * rows - 1) * (2 * cols - 1)
        nbytes += (8 if case.get("dtype") == "float64" else 4) * ((n + m) * rows * cols + k * out)
        if case["method"] in FFT_METHODS:  # real transforms of every matrix and result, products between
            flops += (n + m + k) * 2.5 * out * math.log2(out) + k * 3 * out
        else:
            flops += 2 * k * (rows * cols) ** 2
    return {"bytes": nbytes, "flops": flops}


def definition64(left, right):
    """Every right against one left by the definition, in float64: one matrix product per dy."""
    rows, cols = left.shape
    wide = torch.zeros(rows, 3 * cols - 2, dtype=torch.float64, device=left.device)
    wide[:, cols - 1:2 * cols - 1] = left
    windows = wide.unfold(1, cols, 1)  # [r][dx][c] = left[r][c + dx]
    out = torch.empty(right.shape[0], 2 * rows - 1, 2 * cols - 1, dtype=torch.float64, device=left.device)
    for dy in range(-(rows - 1), rows):
        a, b = max(0, dy), min(rows, rows + dy)
        shifted = windows[a:b].permute(0, 2, 1).reshape((b - a) * cols, 2 * cols - 1)
        out[:, dy + rows - 1] = right[:, a - dy:b - dy].reshape(right.shape[0], -1) @ shifted
    return out


def transform64(left, right):
    """Every right against one left through float64 transforms; beside float32 results exact."""
    rows, cols = left.shape
    size = tuple(1 << (2 * v - 1).bit_length() for v in (rows, cols))
    spectrum = torch.fft.rfft2(left, s=size)
    out = torch.empty(right.shape[0], 2 * rows - 1, 2 * cols - 1, dtype=torch.float64, device=left.device)
    for k in range(right.shape[0]):
        full = torch.fft.irfft2(spectrum * torch.fft.rfft2(right[k], s=size).conj(), s=size)
        out[k] = torch.roll(full, (rows - 1, cols - 1), (0, 1))[:2 * rows - 1, :2 * cols - 1]
    return out


def exact(case, seed):
    left, right = (v.double() for v in inputs(case, seed))
    if case["method"] == "batch":
        _, pairs, _, _, length = batch_layout(case)
        out = torch.empty(length, dtype=torch.float64, device="cuda")
        for lo, ro, oo, rows, cols in pairs:
            got = transform64(left[lo:lo + rows * cols].view(rows, cols), right[ro:ro + rows * cols].view(1, rows, cols))
            out[oo:oo + got.numel()] = got.reshape(-1)
        return out
    one = definition64 if case["dtype"] == "float64" else transform64
    if case["family"] == "n_to_m":
        return torch.cat([one(v, right) for v in left])
    if case["family"] == "n_to_mn":  # result k pairs right k with left k mod n
        n, out = case["n"], None
        for i in range(n):
            got = one(left[i], right[i::n].contiguous())
            out = torch.empty((case["m"],) + got.shape[1:], dtype=torch.float64, device="cuda") if out is None else out
            out[i::n] = got
        return out
    return one(left[0], right)
