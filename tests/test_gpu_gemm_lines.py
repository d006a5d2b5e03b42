"""Sketch products (Y^T = Omega^T A^T, Nl rows, m columns, K = n) on both sides of the lines at which
the kernel that streams A takes over from the tiled ones, with chunk numbers of every remainder by
eight, against an FP64 product of the same values: elementwise K eps (|A| |Omega|), which every
summation order meets.  And two places where the wrong side had been taken, by their times: FP64
products of an even number of rows from 114 to 126 with a long K, and FP32 products with few rows and a
short K."""
import time

import numpy as np
import pytest

from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu

F64 = [(32, 256, 1024), (33, 256, 32767), (40, 256, 32768), (64, 257, 4590), (64, 300, 3932),
       (64, 301, 3932), (48, 1153, 1024), (114, 1030, 32770), (126, 300, 32768), (127, 2048, 32768),
       (128, 2047, 32768), (128, 2050, 32770), (100, 9000, 127), (97, 16384, 128), (96, 16384, 127)]
F32 = [(16, 1151, 1024), (16, 1153, 1024), (17, 512, 9215), (32, 512, 9216), (32, 513, 6131),
       (24, 3073, 1024), (33, 12287, 1024), (48, 12289, 1024), (40, 3074, 4099), (49, 8193, 4096),
       (64, 8190, 4096), (64, 30001, 1120)]


def product(torch, m, n, Nl, dt, ordera):
    gen = torch.Generator(device="cuda").manual_seed(m + n + Nl)
    shape = (m, n) if ordera == "R" else (n, m)
    a = torch.randn(shape, generator=gen, device="cuda", dtype=dt)
    om = torch.randn(n, Nl, generator=gen, device="cuda", dtype=dt)
    return a, om, lambda: pipeline.sketch(capi.create_param(m, n, Nl, 0, 1), a, omega=om, ordera=ordera)


@pytest.mark.parametrize("ordera", ["R", "C"])
@pytest.mark.parametrize("dtype,Nl,m,n", [("float64", *s) for s in F64] +
                         [("float32", *s) for s in F32])
def test_both_sides_of_the_lines(torch_cuda, ordera, dtype, Nl, m, n):
    a, om, run = product(torch_cuda, m, n, Nl, getattr(torch_cuda, dtype), ordera)
    y = run().double()
    a64 = (a if ordera == "R" else a.t().contiguous()).double()
    ref, mag = a64 @ om.double(), a64.abs() @ om.double().abs()
    worst = ((y - ref).abs() / (n * np.finfo(dtype).eps * mag)).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n", [1024 * c + 5 for c in range(1, 18)])
def test_chunk_numbers(torch_cuda, dtype, n):
    a, om, run = product(torch_cuda, 4099, n, 13, getattr(torch_cuda, dtype), "R")
    y = run().double()
    ref, mag = a.double() @ om.double(), a.double().abs() @ om.double().abs()
    worst = ((y - ref).abs() / (n * np.finfo(dtype).eps * mag)).max().item()
    assert worst <= 1.0, worst


def best_times(torch, runs):
    """The least time of each, taken in turn."""
    best = {}
    for i in range(12):
        for key, run in runs.items():
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(10):
                run()
            torch.cuda.synchronize()
            t = (time.perf_counter() - t0) / 10
            if i > 0:
                best[key] = min(t, best.get(key, t))
    return best


def test_even_row_counts_below_128(torch_cuda):
    """126 rows are no dearer than 127 (they took 1.5 times as long)."""
    f64 = torch_cuda.float64
    t = best_times(torch_cuda, {Nl: product(torch_cuda, 4096, 32768, Nl, f64, "R")[2]
                                for Nl in (126, 127)})
    assert t[126] <= 1.25 * t[127], t


def test_few_rows_short_k(torch_cuda):
    """48 FP32 rows against 400 columns of 1024 values are no dearer than 65 rows, on the same tiles (the
    call took 1.3 times as long on the streaming kernel)."""
    f32 = torch_cuda.float32
    t = best_times(torch_cuda, {Nl: product(torch_cuda, 400, 1024, Nl, f32, "R")[2] for Nl in (48, 65)})
    assert t[48] <= 1.2 * t[65], t
