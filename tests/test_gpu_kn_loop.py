"""The KN loop in one launch against the oracle on the same bases: l at the edges of its 16-column
tiles, Nl at the edges of its 16-row slices, the largest sizes it takes and the first it does not, the Newton-Schulz path and the return for the eigendecomposition."""
import numpy as np
import pytest

import oracle as O
from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu


def bases(m, l, N, spread, seed, far=False):
    """N orthonormal m x l blocks around a common subspace; far: block 0 at 45 degrees from the
    others (Z = about 0.2 I in the first iteration, out of reach of series and Newton-Schulz)."""
    rng = np.random.default_rng(seed)
    q, _ = np.linalg.qr(rng.standard_normal((m, 2 * l)))
    out = []
    for i in range(N):
        c = q[:, :l] + spread / np.sqrt(m) * rng.standard_normal((m, l))
        if far and i > 0:
            c = c + q[:, l:]
        out.append(np.linalg.qr(c)[0])
    return np.concatenate(out, 1)


def check(torch, m, l, N, spread, dtype, seed, far=False):
    qs = bases(m, l, N, spread, seed, far).astype(dtype)
    q, it, _ = O.integrate_kolmogorov_nagumo(qs.astype(np.float64), N)
    prm = capi.create_param(m, 2 * l, l, 0, N)
    g, git, _ = pipeline.integrate(prm, torch.from_numpy(qs).cuda(), "KN")
    g = g.double().cpu().numpy()
    # a few rounding errors per product and iteration, and those of M (sums of m terms)
    tol = 8 * (it + np.sqrt(m)) * np.sqrt(l) * np.finfo(dtype).eps
    err = np.linalg.norm(g - q) / np.linalg.norm(q)
    print(f"l={l} N={N} {np.dtype(dtype).name}: {it} iterations, {err:.1e} (tol {tol:.1e})")
    assert git == it
    assert err <= tol


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("l,N", [(1, 1), (1, 5), (11, 12), (16, 1), (16, 65), (17, 3), (32, 8),
                                 (33, 31), (47, 11), (48, 22), (49, 21), (64, 32), (64, 33),
                                 (65, 7), (80, 25), (81, 13)])
def test_loop_matches_oracle(torch_cuda, l, N, dtype):
    check(torch_cuda, 300, l, N, 0.7, dtype, 10 * l + N)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("l,N", [(16, 4), (29, 9), (64, 6)])
def test_loop_newton_schulz(torch_cuda, monkeypatch, l, N, dtype):
    monkeypatch.setenv("ISVD_KN_NS", "1")
    check(torch_cuda, 260, l, N, 0.7, dtype, 7)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("l", [16, 40])
def test_loop_returns_for_the_eigendecomposition(torch_cuda, l, dtype):
    check(torch_cuda, 256, l, 10, 0.2, dtype, 3, far=True)


def test_loop_maxit(torch_cuda):
    qs = torch_cuda.from_numpy(bases(200, 20, 6, 0.7, 1)).cuda()
    prm = capi.create_param(200, 40, 20, 0, 6)
    _, it, err = pipeline.integrate(prm, qs, "KN", argv=[3, 1e-12])
    assert it == 4 and err > 1e-12
    q1, it1, _ = pipeline.integrate(prm, qs, "KN", argv=[1, 0.0])
    ref, rit, _ = O.integrate_kolmogorov_nagumo(qs.cpu().numpy(), 6, maxit=1, tol=0.0)
    assert it1 == rit == 2
    assert np.abs(q1.cpu().numpy() - ref).max() < 1e-13
