"""The Gram and triangular products of CholeskyQR2 at the edges of their register layouts: widths
around multiples of 16 (column tiles) and of a 16-byte vector, row counts around a wave's 16 rows
and a Gram chunk, the smallest m (= l), odd row strides (N l odd), one and several blocks, against
numpy's QR of the same values.

Tolerances: |Q^T Q - I| <= c u (m + l) sqrt(l) after the second pass with c = 30, and Q itself to
kappa (at most about 1e3 for square Gaussian blocks whose columns are scaled by up to 2^3, which a
small ridge keeps there) times that; an element missed, doubled or misplaced gives errors of the
order of 1."""
import numpy as np
import pytest

from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 5, 3), (3, 3, 1), (4, 64, 2), (5, 129, 3), (15, 15, 2), (16, 16, 1),
          (17, 257, 3), (31, 63, 2), (33, 513, 1), (47, 1000, 3), (49, 128, 2), (64, 64, 5),
          (65, 2049, 1), (81, 300, 3), (96, 97, 2), (97, 640, 1), (112, 1023, 2), (113, 131, 3),
          (127, 127, 1), (127, 4099, 3), (128, 128, 3), (128, 5000, 2)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("l,m,N", SHAPES)
def test_row_block_products(torch_cuda, monkeypatch, l, m, N, dtype):
    torch = torch_cuda
    monkeypatch.setenv("ISVD_CHOLQR", "1")
    rng = np.random.default_rng(1000 * l + m)
    y = rng.standard_normal((m, l * N))
    for i in range(N):
        y[:l, i * l:(i + 1) * l] += 4 * np.sqrt(l) * np.eye(l)
    y = (y * np.exp2(rng.uniform(-1.5, 1.5, size=(1, l * N)))).astype(dtype)
    p = capi.create_param(m, m, l, 0, N)
    yd = torch.from_numpy(y).cuda()
    pipeline.orthogonalize(p, yd, "TS")
    q = yd.double().cpu().numpy()
    tol = 30 * np.finfo(dtype).eps * (m + l) * np.sqrt(l)
    for i in range(N):
        qi = q[:, i * l:(i + 1) * l]
        qn, r = np.linalg.qr(y[:, i * l:(i + 1) * l].astype(np.float64))
        assert np.abs(qi.T @ qi - np.eye(l)).max() < tol
        # R has a positive diagonal, which fixes Q itself, not its span alone
        assert np.abs(qi - qn * np.sign(np.diag(r))).max() < 10 * tol
