"""The products of a hierarchical reduction at the edges of their layouts -- B_i = Q_i^T Q_{i+h} (two
tall row-major blocks) and the update W_i^T Q_i^T + T_i^T Q_{i+h}^T (a short K, with and without
accumulation) -- against the oracle on the same bases, and the short-K product as the backward pass
uses it (all of dA) against an FP64 reference.

Tolerance: each of the log2(N) levels multiplies and normalizes by factors of at most 1 and rounds l + m
terms per product: (levels + 1) sqrt(m + l) 8 u with well-separated bases, relative to the unit-norm
projector entries; a misplaced tile or a dropped row gives errors of the order of 1."""
import numpy as np
import pytest

import oracle as O
from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("l,m,N", [(1, 70001, 2), (2, 40000, 3), (3, 30000, 2), (4, 20011, 4),
                                   (5, 16000, 2), (15, 6000, 3), (16, 4096, 2), (17, 5003, 4),
                                   (31, 2200, 2), (33, 2049, 3), (47, 1500, 2), (48, 1400, 5),
                                   (49, 1401, 2), (61, 1100, 4), (64, 1024, 3), (65, 1100, 2),
                                   (96, 900, 3), (97, 1000, 2), (128, 777, 4), (64, 511, 2)])
def test_hierarchical_reduction_products(torch_cuda, l, m, N, dtype):
    rng = np.random.default_rng(l * 7 + m)
    q, _ = np.linalg.qr(rng.standard_normal((m, l)))
    qs = np.concatenate([np.linalg.qr(q + 0.3 / np.sqrt(m) * rng.standard_normal((m, l)))[0]
                         for _ in range(N)], 1).astype(dtype)
    ref = O.integrate_hierarchical_reduction(qs.astype(np.float64), N)
    prm = capi.create_param(m, max(2 * l, 2), l, 0, N)
    g = pipeline.integrate(prm, torch_cuda.from_numpy(qs).cuda(), "HR")
    g = (g[0] if isinstance(g, tuple) else g).double().cpu().numpy()
    ref = ref[0] if isinstance(ref, tuple) else ref
    tol = (np.log2(N) + 2) * 8 * np.sqrt(m + l) * np.finfo(dtype).eps * np.sqrt(l)
    # the basis is fixed up to a rotation: compare the projectors through their action
    x = rng.standard_normal((m, 3))
    assert np.abs(g.T @ g - np.eye(l)).max() < tol
    assert np.linalg.norm(g @ (g.T @ x) - ref @ (ref.T @ x)) < tol * np.linalg.norm(x)
