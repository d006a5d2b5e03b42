"""Sketch products with few columns (Nl <= 64, the kernel that streams A past the matrix cores)
against numpy's FP64 product: rows at the edges of the 16-row tiles, columns at the edges of the
16-byte vectors and of a workgroup's strip, K with and without a checked rest, both storage orders
of A and unaligned views.  The bound is elementwise K eps (|A| |Omega|), which every summation order
meets."""
import numpy as np
import pytest

from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordera", ["R", "C"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("Nl,m,n", [(1, 256, 1024), (15, 257, 1025), (16, 259, 1027),
                                    (17, 1000, 2048), (33, 513, 1031), (48, 300, 4099),
                                    (49, 4097, 1024), (63, 255 + 2, 9001), (64, 2048, 3072)])
@pytest.mark.parametrize("off", [0, 1])
def test_thin_product(torch_cuda, ordera, dtype, Nl, m, n, off):
    torch = torch_cuda
    rng = np.random.default_rng(m + n + Nl)
    a = (rng.standard_normal((m, n)) * np.exp2(rng.integers(-4, 5, size=(m, 1)))).astype(dtype)
    om = rng.standard_normal((n, Nl)).astype(dtype)
    p = capi.create_param(m, n, Nl, 0, 1)
    store = np.ascontiguousarray(a if ordera == "R" else a.T)
    buf = torch.empty(store.size + off, dtype=torch.from_numpy(store).dtype, device="cuda")
    a_arg = buf[off:].view(store.shape)
    a_arg.copy_(torch.from_numpy(store))
    y = pipeline.sketch(p, a_arg, omega=torch.from_numpy(om).cuda(), ordera=ordera)
    y = y.cpu().numpy().astype(np.float64)
    a64, om64 = a.astype(np.float64), om.astype(np.float64)
    err = np.abs(y - a64 @ om64)
    bound = n * np.finfo(dtype).eps * (np.abs(a64) @ np.abs(om64))
    assert (err <= bound).all(), float((err / bound).max())
