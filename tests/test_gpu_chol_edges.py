"""CholeskyQR2's triangular kernel at the edges of its layout: a thread holds 4 x 4 of the block,
so widths around multiples of 4, around one wavefront of tiles (l = 32) and at both ends of its
range (1 and 128), each with several blocks in one launch.

Tolerance: the second pass leaves |Q^T Q - I| <= c u (m + l) sqrt(l) for blocks this well
conditioned; 1e-11 holds that with c = 30 at 700 x 128, and an element missed or taken twice gives
errors of the order of 1."""
import numpy as np
import pytest

from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("l", [1, 2, 3, 4, 5, 7, 8, 9, 31, 32, 33, 61, 64, 65, 127, 128])
def test_cholesky_kernel_edges(torch_cuda, monkeypatch, l):
    torch = torch_cuda
    monkeypatch.setenv("ISVD_CHOLQR", "1")
    m, N = 700, 3
    rng = np.random.default_rng(l)
    y = rng.standard_normal((m, l * N)) * np.exp2(rng.uniform(-3, 3, size=(1, l * N)))
    p = capi.create_param(m, m, l, 0, N)
    yd = torch.from_numpy(y).cuda()
    pipeline.orthogonalize(p, yd, "TS")
    q = yd.cpu().numpy()
    for i in range(N):
        qi = q[:, i * l:(i + 1) * l]
        qn, r = np.linalg.qr(y[:, i * l:(i + 1) * l])
        assert np.abs(qi.T @ qi - np.eye(l)).max() < 1e-11
        # R has a positive diagonal, which fixes Q itself, not its span alone
        assert np.abs(qi - qn * np.sign(np.diag(r))).max() < 1e-10
