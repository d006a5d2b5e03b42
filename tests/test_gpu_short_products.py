"""The outer product dA = Pt^T Rt of the backward pass (K = l + k, a large C) at the edges of its layout:
K around multiples of 16, of a 16-byte vector and around the largest it takes (64), the general path
on either side, row and column counts around the blocks, few rows and few columns, both storage
orders -- against the closed form for a matrix of rank l with an exact Qbar, where the complement has no
singular values: dense_svd_grad over the l triplets plus U_k S_k^-1 gV^T (I - V V^T).

Tolerance: singular values 3 - 2 i / l have gaps of 2 / l, which amplify roundings by about l:
200 l u normwise; one misplaced 16 x 16 tile in 2^24 elements gives 4e-3."""
import numpy as np
import pytest

from adjoint_ref import dense_svd_grad
from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,k,p", [(4099, 4100, 1, 1), (4100, 4099, 1, 2), (262147, 66, 5, 6),
                                     (66, 262147, 5, 7), (4100, 4097, 8, 1), (70001, 257, 16, 16),
                                     (5000, 3501, 20, 23), (4111, 4100, 21, 22),
                                     (4099, 4100, 22, 21)])
@pytest.mark.parametrize("ordera", ["R", "C"])
def test_outer_product_of_the_backward(torch_cuda, ordera, m, n, k, p, dtype):
    torch = torch_cuda
    l = k + p
    g = torch.Generator(device="cuda").manual_seed(m + k)
    rnd = lambda *sh: torch.randn(*sh, generator=g, device="cuda", dtype=torch.float64)
    u, v = torch.linalg.qr(rnd(m, l))[0], torch.linalg.qr(rnd(n, l))[0]
    s = 3 - 2 * torch.arange(l, device="cuda", dtype=torch.float64) / l
    w, GU, GV = rnd(k), rnd(m, k), rnd(n, k)
    dt = torch.float64 if dtype == np.float64 else torch.float32
    a = (u * s) @ v.t()
    a = (a if ordera == "R" else a.t()).to(dt).contiguous()
    prm = capi.create_param(m, n, k, p, 1)
    qbar = u.to(dt).contiguous()
    kw = {} if ordera == "R" else {"ordera": "C"}
    da = pipeline.isvd_backward(prm, a, qbar, w.to(dt), GU.to(dt).contiguous(),
                                GV.to(dt).contiguous(), "GR", **kw).double()
    _, uf, _ = pipeline.postprocess(prm, a, qbar, "GR", **kw)
    sg = torch.sign((uf.double()[:, :k] * u[:, :k]).sum(0))
    u, v = u.clone(), v.clone()
    u[:, :k] *= sg
    v[:, :k] *= sg
    ref = dense_svd_grad(torch, u, s, v, w, GU, GV, k)
    ref = ref + (u[:, :k] / s[:k]) @ (GV.t() - (GV.t() @ v) @ v.t())
    if ordera == "C" and da.shape != ref.shape:
        da = da.t()
    err = ((da - ref).norm() / ref.norm()).item()
    assert err < 200 * l * np.finfo(dtype).eps, err
