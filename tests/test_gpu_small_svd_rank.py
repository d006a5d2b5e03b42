"""The l x l SVD and PSD eigendecomposition on columns that collapse onto each other (rank one, equal
and zero columns, rank-one diagonal blocks) or differ by many orders of magnitude, through the entry
points, against numpy's singular values of the same matrix."""
import numpy as np
import pytest

from isvd_amd import capi, pipeline

pytestmark = pytest.mark.gpu

M, NCOL = 200, 160  # B = Qbar^T A is l x 160; Qbar = the first l coordinate vectors


def rank_one(l, rng):
    return np.outer(rng.standard_normal(l), rng.standard_normal(NCOL))


def equal(l, rng):  # rank 3, rows that repeat exactly
    return rng.integers(-2, 3, (l, 3)).astype(float) @ rng.standard_normal((3, NCOL))


def blocks(l, rng):  # rank-one blocks on the diagonal
    b, size = np.zeros((l, NCOL)), max(2, l // 4)
    for i, r0 in enumerate(range(0, l, size)):
        r = min(size, l - r0)
        b[r0:r0 + r, 20 * (i % 8):20 * (i % 8) + 20] = np.outer(rng.standard_normal(r),
                                                                rng.standard_normal(20))
    return b


def zeros(l, rng):  # zero rows between dense ones, more at the end
    b = rng.standard_normal((l, NCOL))
    b[::2] = 0
    b[3 * l // 4:] = 0
    return b


def scaled(l, rng):  # rows from 1 down to 1e-15
    return rng.standard_normal((l, NCOL)) * 10.0 ** (-15 * np.arange(l)[:, None] / (l - 1))


FAMILIES = {f.__name__: f for f in (rank_one, equal, blocks, zeros, scaled)}
FAMILIES["ones"] = lambda l, rng: np.ones((l, NCOL))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("alg", ["GR", "TS"])
@pytest.mark.parametrize("family", sorted(FAMILIES))
@pytest.mark.parametrize("l", [4, 12, 32, 47, 64, 128])
def test_postprocess(torch_cuda, l, family, alg, dtype):
    torch = torch_cuda
    b = FAMILIES[family](l, np.random.default_rng(l)).astype(dtype)
    a = np.zeros((M, NCOL), dtype)
    a[:l] = b
    ref = np.linalg.svd(b.astype(np.float64), compute_uv=False)
    s, u, v = (t.double().cpu().numpy() for t in pipeline.postprocess(
        capi.create_param(M, NCOL, l, 0, 1), torch.from_numpy(a).cuda(),
        torch.from_numpy(np.eye(M, l, dtype=dtype)).cuda(), alg))
    # the Gramian halves the digits of what lies below sqrt(eps)
    tol = 40 * l * np.finfo(dtype).eps
    assert np.isfinite(s).all()
    assert np.abs(s - ref).max() <= (tol if alg == "TS" else np.sqrt(tol)) * ref[0]
    big = int((ref > 1e-2 * ref[0]).sum())
    assert np.abs(s - ref)[:big].max() <= tol * (1 if alg == "TS" else 1e2) * ref[0]
    assert np.isfinite(u[:, :big]).all() and np.isfinite(v[:, :big]).all()
    r = a - (u[:, :big] * s[:big]) @ v[:, :big].T
    assert np.linalg.norm(r) <= np.linalg.norm(ref[big:]) + tol * np.sqrt(l) * ref[0] * (
        1 if alg == "TS" else 1e2)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("l", [12, 32, 64, 128])
def test_hierarchical_reduction_of_overlapping_bases(torch_cuda, l, dtype):
    """Two bases that share one direction only: Q_0^T Q_1 is of rank one."""
    torch = torch_cuda
    q = np.linalg.qr(np.random.default_rng(l).standard_normal((300, 2 * l)))[0]
    q0, q1 = q[:, :l], np.concatenate([q[:, :1], q[:, l + 1:]], 1)
    x = np.linalg.qr(np.random.default_rng(1).standard_normal((l, l)))[0]
    qs = np.concatenate([q0 @ x, q1 @ x.T], 1).astype(dtype)
    g, _, _ = pipeline.integrate(capi.create_param(300, 2 * l, l, 0, 2),
                                 torch.from_numpy(qs).cuda(), "HR")
    g = g.double().cpu().numpy()
    tol = 40 * l * np.finfo(dtype).eps
    assert np.isfinite(g).all()
    # the shared direction is in the result, and the columns are orthonormal
    assert np.linalg.norm(q[:, 0] - g @ (g.T @ q[:, 0])) <= tol
    assert np.abs(g.T @ g - np.eye(l)).max() <= tol


def test_hierarchical_reduction_memory(torch_cuda):
    """The rotation logs of a level's SVDs (320 of 128 x 128 here) stay within 640 MB: the pool's high
    water mark, beside the right result."""
    import ctypes
    torch = torch_cuda
    hip = ctypes.CDLL("libamdhip64.so")
    l, N = 128, 640
    q = np.linalg.qr(np.random.default_rng(0).standard_normal((160, l)))[0]
    x = np.linalg.qr(np.random.default_rng(1).standard_normal((N, l, l)))[0]
    qs = torch.from_numpy(np.concatenate(list(q @ x), 1)).cuda()
    prm = capi.create_param(160, 150, l, 0, N)
    pipeline.integrate(capi.create_param(160, 150, 8, 0, 2), qs[:, :16].clone(), "HR")
    pool, high, zero = ctypes.c_void_p(), ctypes.c_uint64(), ctypes.c_uint64(0)
    assert hip.hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0
    used_mem_current, used_mem_high = 7, 8  # hipMemPoolAttr
    assert hip.hipMemPoolSetAttribute(pool, used_mem_high, ctypes.byref(zero)) == 0
    assert hip.hipMemPoolGetAttribute(pool, used_mem_current, ctypes.byref(high)) == 0
    before = high.value
    g, _, _ = pipeline.integrate(prm, qs, "HR")
    assert hip.hipMemPoolGetAttribute(pool, used_mem_high, ctypes.byref(high)) == 0
    assert high.value > before
    # B, W, T and S of every pair and the merged bases: 320 problems
    others = (N // 2) * (3 * l * l + l + 160 * l) * 8
    assert high.value - before <= (640 << 20) + others + (64 << 20)
    g = g.cpu().numpy()
    tol = 40 * l * np.finfo(float).eps
    assert np.abs(g.T @ g - np.eye(l)).max() <= tol
    assert np.linalg.norm(g - q @ (q.T @ g)) <= tol
