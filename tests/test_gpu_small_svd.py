"""The l x l SVD and PSD eigendecomposition behind the postprocessing, through its entry points, at
the edges of the Jacobi kernel's groups of four columns and 16-row padding: singular values, both
singular bases and the reconstruction, for graded, clustered, rank-deficient and diagonal spectra."""
import numpy as np
import pytest

from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu

SPECTRA = {
    "graded": lambda l: 10.0 ** (-5.0 * np.arange(l) / max(l - 1, 1)),
    "clustered": lambda l: np.where(np.arange(l) < (l + 1) // 2, 1.0, 0.5),
    "deficient": lambda l: np.where(np.arange(l) < max(1, l - 3), 0.9 ** np.arange(l), 0.0),
}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("alg", ["TS", "GR"])
@pytest.mark.parametrize("spec", sorted(SPECTRA))
@pytest.mark.parametrize("l", [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 48, 63, 64, 65, 100, 127, 128])
def test_postprocess_svd(torch_cuda, l, spec, alg, dtype):
    torch = torch_cuda
    m, n = 200, 150
    rng = np.random.default_rng(l)
    sv = SPECTRA[spec](l)
    q = np.linalg.qr(rng.standard_normal((m, l)))[0]
    x = np.linalg.qr(rng.standard_normal((l, l)))[0]
    v = np.linalg.qr(rng.standard_normal((n, l)))[0]
    a = ((q @ x) * sv) @ v.T
    qd = torch.from_numpy(q.astype(dtype)).cuda()
    ad = torch.from_numpy(a.astype(dtype)).cuda()
    s, u, w = (t.double().cpu().numpy() for t in
               pipeline.postprocess(capi.create_param(m, n, l, 0, 1), ad, qd, alg))
    eps = np.finfo(dtype).eps
    # the Gramian halves the digits of what lies below sqrt(eps)
    tol = 40 * l * eps
    s_tol = tol if alg == "TS" else np.sqrt(tol)
    assert (np.diff(s) <= 0).all()
    big = sv > 1e-2
    assert np.abs(s - sv)[big].max() <= tol * (1 if alg == "TS" else 1e2)
    assert np.abs(s - sv).max() <= s_tol
    k = int(big.sum())
    for z in (u, w):
        g = z[:, :k].T @ z[:, :k]
        assert np.abs(g - np.eye(k)).max() <= tol * (1 if alg == "TS" else 1e4)
    # A - U S V^T is what the basis leaves out (nothing) and rounding
    r = a - (u[:, :k] * s[:k]) @ w[:, :k].T
    left = np.linalg.norm(sv[k:])
    assert np.linalg.norm(r) <= left + tol * np.sqrt(l) * (1 if alg == "TS" else 1e2)
    if alg == "TS" and spec != "deficient":
        g = w.T @ w
        assert np.abs(g - np.eye(l)).max() <= tol


def test_zero_matrix(torch_cuda):
    torch = torch_cuda
    q = torch.linalg.qr(torch.randn(100, 20, device="cuda", dtype=torch.float64))[0].contiguous()
    a = torch.zeros(100, 60, device="cuda", dtype=torch.float64)
    s, _, _ = pipeline.postprocess(capi.create_param(100, 60, 20, 0, 1), a, q, "GR", want_v=False)
    assert (s == 0).all()
