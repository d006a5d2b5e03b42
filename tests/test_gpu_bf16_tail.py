"""BF16 products whose last round of tiles is cut in K: a few tiles past one round, tile rows and columns
that end inside a tile, K with a partial step, whole rounds (nothing cut), through the sketch against
the FP64 product of the same values within the FP32 accumulation bound (n / 16 + 32) u sum |a||b| (a cut
adds at most 16 roundings, as split-K does); and the Gram product with its skipped half through the
mixed KN integration against the FP64 one on the same bases (same bars as the workload-size test)."""
import numpy as np
import pytest

from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordera", ["C", "R"])
@pytest.mark.parametrize("m,n,l,N", [(4099, 2100, 100, 43), (7681, 4100, 128, 20),
                                     (6400, 8192, 64, 44), (5121, 20000, 125, 40),
                                     (8192, 2048, 128, 32)])
def test_sketch_tail(torch_cuda, ordera, m, n, l, N):
    torch = torch_cuda
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    shape = (m, n) if ordera == "R" else (n, m)
    a = torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)
    om = torch.randn(n, N * l, generator=gen, device="cuda").to(torch.bfloat16)
    y = pipeline.sketch(capi.create_param(m, n, l, 0, N), a, omega=om, ordera=ordera).double()
    a64 = (a if ordera == "R" else a.t().contiguous()).double()
    ref, mag = a64 @ om.double(), a64.abs() @ om.double().abs()
    bound = (n / 16 + 32) * 2.0 ** -24 * mag
    assert ((y - ref).abs() <= bound).all().item()


def test_gram_tail(torch_cuda):
    torch = torch_cuda
    m, l, N = 49152, 128, 32
    gen = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda: torch.randn(m, l, generator=gen, device="cuda", dtype=torch.float64)
    q = torch.linalg.qr(rnd())[0]
    qs = torch.cat([torch.linalg.qr(q + 0.7 / m ** 0.5 * rnd())[0] for _ in range(N)], 1)
    p = capi.create_param(m, 2 * l, l, 0, N)
    q64, it64, _ = pipeline.integrate(p, qs, "KN", [256, 1e-4])
    q32, it32, _ = pipeline.integrate(p, qs.float(), "KN", [256, 1e-4], mixed=True)
    assert abs(it32 - it64) <= 1
    # sines of the angles between the two subspaces
    r = q32.double() - q64 @ (q64.t() @ q32.double())
    assert torch.linalg.norm(r, 2).item() < 1e-4
