"""Products of more than 64 rows whose operands go straight to the matrix cores, through the sketch
(Y^T = Omega^T A^T, with Nl rows, m columns and K = n) against an FP64 product of the same values: rows
at the edges of the 16-row tiles and of the 48- and 64-row blocks (one row past a block, a block short
of a vector), columns at the edges of the vectors and strips, K with and without a rest and cut into
chunks, both storage orders, unaligned views, strips of one and of two column sets; the products just
below the line, which the tiled kernels take; and the symmetric product through the KN integration.

The bound of a product is elementwise K eps (|A| |Omega|), which every summation order meets; the KN
bound is a few rounding errors per product and iteration plus those of M's sums of m terms."""
import numpy as np
import pytest

import oracle as O
from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu

# Nl = N l rows, m columns, K = n
F64 = [(1, 65, 1000, 1024), (1, 66, 771, 1031), (1, 67, 12289, 64 + 3), (1, 80, 5000, 129),
       (1, 96, 801, 700), (1, 113, 300, 1537), (1, 127, 257, 2050), (1, 128, 129, 32768 + 5),
       (1, 128, 66, 40000), (3, 43, 1001, 1000), (11, 47, 1001, 301), (16, 32, 2000, 1000),
       (4, 50, 513, 511), (4, 65, 16501, 8100), (1, 65, 999, 700)]
F32 = [(1, 113, 75001, 1030), (3, 43, 13003, 5150), (11, 47, 10007, 1700), (4, 65, 16385, 2100),
       (16, 32, 16384, 1024), (3, 64, 8191, 5500), (2, 100, 3000, 2000)]


@pytest.mark.parametrize("ordera", ["R", "C"])
@pytest.mark.parametrize("dtype,N,l,m,n", [("float64", *s) for s in F64] +
                         [("float32", *s) for s in F32])
def test_stream_product(torch_cuda, ordera, dtype, N, l, m, n):
    torch = torch_cuda
    dt = getattr(torch, dtype)
    off = (m + l) % 2  # an element past an allocation's alignment
    gen = torch.Generator(device="cuda").manual_seed(m + n + l)
    shape = (m, n) if ordera == "R" else (n, m)
    a = torch.empty(m * n + off, dtype=dt, device="cuda")[off:].view(shape)
    a.copy_(torch.randn(shape, generator=gen, device="cuda", dtype=dt))
    om = torch.randn(n, N * l, generator=gen, device="cuda", dtype=dt)
    p = capi.create_param(m, n, l, 0, N)
    y = pipeline.sketch(p, a, omega=om, ordera=ordera).double()
    a64 = (a if ordera == "R" else a.t().contiguous()).double()
    ref, mag = a64 @ om.double(), a64.abs() @ om.double().abs()
    worst = ((y - ref).abs() / (n * np.finfo(dtype).eps * mag)).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("dtype,m,l,N", [("float64", 1003, 47, 5), ("float64", 300, 65, 7),
                                         ("float32", 7741, 48, 22), ("float32", 3000, 65, 26)])
def test_stream_symmetric_product(torch_cuda, dtype, m, l, N):
    rng = np.random.default_rng(m)
    q, _ = np.linalg.qr(rng.standard_normal((m, l)))
    qs = np.concatenate([np.linalg.qr(q + 0.7 / np.sqrt(m) * rng.standard_normal((m, l)))[0]
                         for _ in range(N)], 1).astype(dtype)
    ref, it, _ = O.integrate_kolmogorov_nagumo(qs.astype(np.float64), N)
    prm = capi.create_param(m, 2 * l, l, 0, N)
    g, git, _ = pipeline.integrate(prm, torch_cuda.from_numpy(qs).cuda(), "KN")
    g = g.double().cpu().numpy()
    assert git == it
    tol = 8 * (it + np.sqrt(m)) * np.sqrt(l) * np.finfo(dtype).eps
    assert np.linalg.norm(g - ref) <= tol * np.linalg.norm(ref)
