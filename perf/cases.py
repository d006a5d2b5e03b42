"""The work this framework is used for, as measurable cases.

A case is one call (or one forward + backward) through the public Python entry points of
``isvd_amd.pipeline`` / ``isvd_amd.autograd``, on a synthetic matrix A = U diag(s) V^T + noise
whose spectrum decays to a tenth of its first value at the requested rank (so that the rank-k
triplets are determined well enough to be compared element by element), at the sizes of this
repository's own workloads: the reference's 101 x 1001 fixture, the 2000 x 1000 demo, the
131072 x 16384 headline, the 65536 x 8192 differentiation workload, and ordinary and ragged
sizes between them.

Wen-Yin integration is not among them: it stops at a loose gradient tolerance after a line search
that amplifies rounding (two runs of the reference algorithm on bases that differ in the last bit
stop at different points), so its outputs cannot be compared value by value.

Singular vectors are defined up to a sign, which a caller fixes for itself (the largest entry of
each right vector made positive), as here in ``_signed``.
"""
import math

import numpy as np
import torch

from isvd_amd import autograd, capi, pipeline

_F64 = torch.float64
_STORED = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16,
           "fp8": torch.float32}


def _case(name, op, dtype, m, n, k, p, N, order="R", orth="TS", integ="KN", post="TS",
          host=False, sym=False):
    c = {"op": op, "dtype": dtype, "m": m, "n": n, "k": k, "p": p, "N": N, "order": order,
         "orth": orth, "integ": integ, "post": post, "host": host, "sym": sym}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the reference's test fixture: the smallest call, all launch and synchronization latency
        _case("fixture_f64_101x1001", "isvd", "f64", 101, 1001, 8, 3, 12, "C", "GR", "KN", "GR"),
        # the reference's demo program: a small decomposition, KN iterations of a few launches
        _case("demo_f64_2000x1000", "isvd", "f64", 2000, 1000, 20, 12, 16, "C", "GR", "KN", "GR"),
        # a C caller's host arrays in and out (the reference's only kind of argument)
        _case("host_f64_4096x1024", "isvd", "f64", 4096, 1024, 20, 12, 16, "C", host=True),
        # ragged everything: odd sizes, odd leading dimensions, a data matrix as it comes
        _case("ragged_f64_10007x3001", "isvd", "f64", 10007, 3001, 37, 10, 11, "R", "TS", "KN",
              "GR"),
        # an ordinary single-precision decomposition of a row-major (torch-like) matrix
        _case("ordinary_f32_16384x4096", "isvd", "f32", 16384, 4096, 20, 12, 16, "R"),
        # hierarchical reduction in place of the iteration
        _case("hr_f64_8192x2048", "isvd", "f64", 8192, 2048, 50, 14, 8, "C", "TS", "HR", "TS"),
        # a symmetric matrix (kernel / covariance matrix) with symmetric postprocessing
        _case("symmetric_f64_4096", "isvd", "f64", 4096, 4096, 20, 12, 8, "C", "GR", "KN", "SY",
              sym=True),
        # new data against a kept basis: the postprocessing stage alone
        _case("project_f64_32768x8192", "post", "f64", 32768, 8192, 32, 16, 1, "R", post="GR"),
        # differentiation through the decomposition: forward (stage by stage) and backward
        _case("train_f32_65536x8192", "train", "f32", 65536, 8192, 16, 16, 16, "R"),
        # the BF16 family at the headline shape
        _case("mixed_bf16_131072x16384", "isvd", "bf16", 131072, 16384, 100, 28, 32, "C", "GR",
              "KN", "TS"),
        # the FP8 family: quantization (encode) and decomposition of a large matrix
        _case("fp8_131072x16384", "isvd", "fp8", 131072, 16384, 64, 64, 32, "R", "GR", "KN", "TS"),
        # the headline: FP64 at 131072 x 16384
        _case("headline_f64_131072x16384", "isvd", "f64", 131072, 16384, 100, 28, 32, "C"),
    ]


# the most m n N l a drawn case takes, by type (each below the listed case of its type or of the
# next dearer one)
_MOST = {"f64": 1.0e12, "f32": 1.6e12, "bf16": 8.0e12, "fp8": 8.0e12}


def draw(rng):
    """One more case: any family and option of the listed ones, sizes over their whole range."""
    def size(lo, hi):
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        how = rng.random()
        if how < 0.4:
            v |= 1
        elif how < 0.7 and v >= 128:
            v -= v % 64
        return max(lo, min(hi, v))

    while True:
        op = rng.choice(["isvd"] * 8 + ["post", "train"])
        dtype = {"post": "f64", "train": "f32"}.get(op) or rng.choice(
            ["f64", "f64", "f64", "f32", "f32", "bf16", "bf16", "fp8"])
        m, n = size(100, 131072), size(100, 16384)
        # single precision resolves fewer neighbouring singular values
        k = size(5, 100 if dtype != "f32" else 20 if op == "isvd" else 16)
        p = rng.randint(3, 28 if dtype != "f32" else 12)
        N = 1 if op == "post" else rng.randint(2, 32)
        integ = "HR" if dtype == "f64" and op == "isvd" and rng.random() < 0.15 else "KN"
        sym = dtype == "f64" and op == "isvd" and integ == "KN" and rng.random() < 0.1
        if sym:
            m = n
        l = k + p
        if l > 128 or 4 * l > min(m, n):
            continue
        if m * n * max(N, 16) * l > _MOST[dtype] or (op == "train" and m * n > 1 << 28):
            continue
        host = (not sym and dtype == "f64" and op == "isvd" and m * n <= 1 << 23
                and rng.random() < 0.3)
        post = "SY" if sym else "TS" if dtype == "f32" else rng.choice(["TS", "GR"])
        orth = rng.choice(["TS", "GR"]) if op == "isvd" else "TS"
        order = "R" if op == "train" else rng.choice(["R", "C"])
        return _case(None, op, dtype, m, n, k, p, N, order, orth, integ, post, host, sym)


# ---- inputs ------------------------------------------------------------------------------------

def _basis(x):
    """An orthonormal basis of x's columns, with its triangular factor: x = q r (CholeskyQR2)."""
    eye, r = torch.eye(x.shape[1], device=x.device, dtype=x.dtype), None
    for _ in range(2):
        c = torch.linalg.cholesky(x.T @ x)
        x = x @ torch.linalg.solve_triangular(c, eye, upper=False).T.contiguous()
        r = c.T if r is None else c.T @ r
    return x, r


def _orthonormal(rows, r, gen):
    return _basis(torch.randn(rows, r, generator=gen, device="cuda", dtype=_F64))[0]


def _matrix(case, seed):
    """A in the storage the entry points take: row-major m x n ('R') or n x m, A^T ('C')."""
    m, n, k, l = case["m"], case["n"], case["k"], case["k"] + case["p"]
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    r = min(4 * l, min(m, n) // 2)
    u = _orthonormal(m, r, gen)
    v = u if case["sym"] else _orthonormal(n, r, gen)
    i = torch.arange(r, device="cuda", dtype=_F64)
    if case["op"] == "train":
        s, noise = 2 * 0.9 ** i + 0.01, 0.01 / (math.sqrt(m) + math.sqrt(n))
    else:
        s, noise = 0.1 ** (i / k), 1e-6
    us = u * s
    c = case["order"] == "C"
    a = torch.empty((n, m) if c else (m, n), device="cuda", dtype=_STORED[case["dtype"]])
    for r0 in range(0, m, 16384):
        t = us[r0:r0 + 16384] @ v.T
        if not case["sym"]:
            t.add_(torch.randn(t.shape, generator=gen, device="cuda"), alpha=noise)
        if c:
            a[:, r0:r0 + t.shape[0]].copy_(t.T)
        else:
            a[r0:r0 + t.shape[0]].copy_(t)
    return a, gen


def _extra(case, gen):
    """What the call takes beside A: Omega and the outputs' gradients."""
    m, n, k, l = case["m"], case["n"], case["k"], case["k"] + case["p"]
    if case["op"] == "train":
        def g(*shape):
            return torch.randn(*shape, generator=gen, device="cuda")
        return {"omega": g(n, case["N"] * l), "gs": g(k), "gu": g(m, k), "gv": g(n, k)}
    return {}


def prepare(case, seed):
    a, gen = _matrix(case, seed)
    st = {"case": case, "a": a, "seed": int(seed) & 0x7FFFFFFF, **_extra(case, gen),
          "prm": capi.create_param(case["m"], case["n"], case["k"], case["p"], case["N"])}
    if case["op"] == "post":
        # the basis that an earlier call on like data left: the range of this one's sketch
        x = _mul(case, a, torch.randn(case["n"], case["k"] + case["p"], generator=gen,
                                      device="cuda", dtype=_F64))
        st["qbar"] = _basis(x)[0]
    if case["dtype"] == "fp8":
        st["a_bf16"] = a.to(torch.bfloat16)
    if case["host"]:
        st["a"] = a.cpu().numpy()
    if case["op"] == "train":
        st["a"].requires_grad_(True)
    return st


# ---- one pass ----------------------------------------------------------------------------------

def _signed(u, v):
    if isinstance(v, np.ndarray):
        g = np.sign(v[np.abs(v).argmax(0), np.arange(v.shape[1])])
    else:
        g = v.gather(0, v.abs().argmax(0, keepdim=True)).sign()[0]
    return u * g, v * g


def run(state):
    c, prm, k = state["case"], state["prm"], state["case"]["k"]
    if c["op"] == "train":
        s, u, v = autograd.isvd(state["a"], state["omega"], k, c["p"], c["N"],
                                ("GP", c["orth"], c["integ"], c["post"]))
        u, v = _signed(u, v)
        da, = torch.autograd.grad((s, u, v), state["a"],
                                  (state["gs"], state["gu"], state["gv"]))
        return {"s": s.detach(), "u": u.detach(), "v": v.detach(), "da": da}
    if c["op"] == "post":
        s, u, v = pipeline.postprocess(prm, state["a"], state["qbar"], c["post"], c["order"])
        u, v = _signed(u[:, :k], v[:, :k])
        return {"s": s, "u": u, "v": v}
    algs = ("GP", c["orth"], c["integ"], c["post"])
    out = {}
    if c["dtype"] == "fp8":
        a8, scale = pipeline.quantize_e4m3(state["a"], c["order"])
        out = {"codes": a8, "scale": scale}
        r = pipeline.isvd_e(prm, a8, scale, state["a_bf16"], seed=state["seed"], algs=algs,
                            ordera=c["order"])
    else:
        r = pipeline.isvd(prm, state["a"], seed=state["seed"], algs=algs, ordera=c["order"])
    u, v = _signed(r["u"][:, :k], r["v"][:, :k])
    return {**out, "s": r["s"], "u": u, "v": v}


# ---- what a pass cannot do without -------------------------------------------------------------

def work(case):
    """Inputs read once, outputs written once, and the products of the method itself (the
    iterations of the integration, whose number the data decides, are left out)."""
    m, n, k, l, N = case["m"], case["n"], case["k"], case["k"] + case["p"], case["N"]
    e = {"f64": 8, "f32": 4, "bf16": 2, "fp8": 4}[case["dtype"]]
    w = 8 if case["dtype"] == "f64" else 4
    nl = N * l
    post_f = 2.0 * m * n * l + 2.0 * n * l * l + 2.0 * (m + n) * l * k
    post_b = w * (l + k * (m + n))
    if case["op"] == "post":
        return {"bytes": e * m * n + w * m * l + post_b, "flops": post_f}
    flops = 2.0 * m * n * nl + 4.0 * m * l * l * N + post_f
    flops += (1.0 * m * nl * nl + 2.0 * m * nl * l) if case["integ"] == "KN" else 6.0 * m * l * nl
    nbytes = e * m * n + post_b
    if case["op"] == "train":
        # the outputs' gradients and dA; A^T X, A Y and the two outer products of dA
        nbytes += w * (m * n + n * nl + k * (m + n))
        flops += post_f + 4.0 * m * n * k + 2.0 * m * n * (l + k)
    if case["dtype"] == "fp8":
        nbytes += 2.0 * m * n + 1.0 * m * n  # the BF16 copy, and the codes written
    return {"bytes": float(nbytes), "flops": flops}


# ---- the same in plain torch, FP64 -------------------------------------------------------------

def _mul(case, a, x):
    """A x in FP64, by row blocks of A."""
    out = torch.empty(case["m"], x.shape[1], device="cuda", dtype=_F64)
    for r0 in range(0, case["m"], 16384):
        t = a[:, r0:r0 + 16384].T if case["order"] == "C" else a[r0:r0 + 16384]
        out[r0:r0 + 16384] = t.to(_F64) @ x
    return out


def _tmul(case, a, x):
    """A^T x in FP64, by row blocks of A."""
    out = torch.zeros(case["n"], x.shape[1], device="cuda", dtype=_F64)
    for r0 in range(0, case["m"], 16384):
        t = a[:, r0:r0 + 16384].T if case["order"] == "C" else a[r0:r0 + 16384]
        out += t.to(_F64).T @ x[r0:r0 + 16384]
    return out


def _omega(seed, n, nl):
    """The seeded Gaussian matrix: Philox-4x32-10 at counter (e, 0, 0, 0), Box-Muller."""
    mask = 0xFFFFFFFF
    out = torch.empty(n * nl, device="cuda", dtype=_F64)
    for e0 in range(0, n * nl, 1 << 24):
        e = torch.arange(e0, min(n * nl, e0 + (1 << 24)), device="cuda", dtype=torch.int64)
        c = [e & mask, e >> 32, torch.zeros_like(e), torch.zeros_like(e)]
        k0, k1 = seed & mask, (seed >> 32) & mask

        def mul(f, x):  # (high, low) 32 bits of a 32 x 32 bit product
            lo, hi = f * (x & 0xFFFF), f * (x >> 16)
            t = (lo >> 16) + hi
            return (t >> 16) & mask, ((t << 16) | (lo & 0xFFFF)) & mask

        for _ in range(10):
            h0, l0 = mul(0xD2511F53, c[0])
            h1, l1 = mul(0xCD9E8D57, c[2])
            c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
            k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
        u1 = (((c[0] << 21) | (c[1] >> 11)) + 1).to(_F64) * 2.0 ** -53
        u2 = (((c[2] << 21) | (c[3] >> 11)) + 1).to(_F64) * 2.0 ** -53
        out[e0:e0 + e.numel()] = torch.sqrt(-2 * torch.log(u1)) * torch.cos(2 * math.pi * u2)
    return out.view(n, nl)


def _dequantized(a32, order):
    """(A as its e4m3 codes stand for it, block scales) of an FP32 matrix, row-major."""
    a = a32.T if order == "C" else a32
    m, n = a.shape
    pad = torch.nn.functional.pad(a, (0, -n % 128, 0, -m % 128))
    blocks = pad.view(pad.shape[0] // 128, 128, pad.shape[1] // 128, 128)
    top = blocks.abs().amax((1, 3)).to(_F64)
    s = torch.exp2(torch.ceil(torch.log2(top / 448)))
    s = torch.where(top > 448 * s, 2 * s, torch.where(top <= 224 * s, s / 2, s))
    s = torch.where(top > 0, s, torch.ones_like(s))
    q = (blocks / s[:, None, :, None].float()).to(torch.float8_e4m3fn).float()
    return (q * s[:, None, :, None].float()).reshape(pad.shape)[:m, :n].contiguous(), s


def _bases(y, N):
    """Orthonormal bases of the N blocks of y, side by side."""
    return torch.cat([_basis(b)[0] for b in y.chunk(N, 1)], 1)


def _kolmogorov_nagumo(qs, N, l, maxit=256, tol=1e-4):
    M = qs.T @ qs
    x = torch.zeros(N * l, l, device="cuda", dtype=_F64)
    x[:l] = torch.eye(l, device="cuda", dtype=_F64)
    b = M @ x
    for _ in range(maxit):
        bg = M @ b / N
        d = b.T @ b / N
        z = b.T @ bg / N - d.T @ d
        w, zv = np.linalg.eigh(((z + z.T) / 2).cpu().numpy())
        sv = np.sqrt(0.5 + np.sqrt(0.25 - w))
        c, ci = (torch.from_numpy((zv * t) @ zv.T).cuda() for t in (sv, 1 / sv))
        f = c - d @ ci
        x, b = x @ f + b @ ci / N, b @ f + bg @ ci
        if np.linalg.norm(sv - 1) <= tol:
            break
    return qs @ x


def _hierarchical(qs, N):
    q, h2 = list(qs.chunk(N, 1)), N
    while h2 > 1:
        h = h2 // 2
        for i in range(h):
            w, s, t = np.linalg.svd((q[i].T @ q[i + h]).cpu().numpy())
            w, s, t = (torch.from_numpy(np.ascontiguousarray(z)).cuda() for z in (w, s, t))
            q[i] = (q[i] @ w + q[i + h] @ t.T) / torch.sqrt(2 * (1 + s))
        h2 = (h2 + 1) // 2
    return q[0]


def _triplets(case, a, q):
    """All l triplets of Q Q^T A (or eigenpairs of Q^T A Q, ascending, for 'SY')."""
    z = _tmul(case, a, q)
    if case["post"] == "SY":
        w = z.T @ q
        s, e = np.linalg.eigh(((w + w.T) / 2).cpu().numpy())
        u = q @ torch.from_numpy(e).cuda()
        return torch.from_numpy(s).cuda(), u, u
    qz, r = _basis(z)
    x, s, yt = np.linalg.svd(r.T.cpu().numpy())  # Z^T = R^T Q_z^T
    x, s, yt = (torch.from_numpy(np.ascontiguousarray(t)).cuda() for t in (x, s, yt))
    return s, q @ x, qz @ yt.T


def _gradient(case, a, s, u, v, gs, gu, gv):
    """dL/dA of the leading k triplets, the discarded part of A entering by its series."""
    k, l = case["k"], case["k"] + case["p"]
    m, n = case["m"], case["n"]
    gup, gvp = torch.zeros(m, l, device="cuda", dtype=_F64), torch.zeros(n, l, device="cuda",
                                                                         dtype=_F64)
    gup[:, :k], gvp[:, :k] = gu, gv
    gsp = torch.zeros(l, device="cuda", dtype=_F64)
    gsp[:k] = gs
    J, K = u.T @ gup, v.T @ gvp
    d = s[None, :] ** 2 - s[:, None] ** 2
    F = torch.where(d == 0, torch.zeros_like(d), 1 / torch.where(d == 0, torch.ones_like(d), d))
    core = (F * (J - J.T)) * s[None, :] + s[:, None] * (F * (K - K.T)) + torch.diag(gsp)

    def proj(x):
        return x - u @ (u.T @ x)

    def ac(y):
        return proj(_mul(case, a, y))

    def act(x):
        return _tmul(case, a, proj(x))

    sk2 = s[:k] ** 2
    xt = proj(gu) / sk2
    yt = (gv - v @ (v.T @ gv)) / sk2
    X, Y = xt.clone(), yt.clone()
    for _ in range(400):
        xt, yt = ac(act(xt)) / sk2, act(ac(yt)) / sk2
        X += xt
        Y += yt
        if max(float(xt.norm() / X.norm()), float(yt.norm() / Y.norm())) < 1e-14:
            break
    E, H = X * s[:k] + ac(Y), act(X) + Y * s[:k]
    return u @ core @ v.T + E @ v[:, :k].T + u[:, :k] @ H.T


def exact(case, seed):
    if case["op"] == "post":
        st = prepare(case, seed)
        s, u, v = _triplets(case, st["a"], st["qbar"])
        u, v = _signed(u[:, :case["k"]], v[:, :case["k"]])
        return {"s": s, "u": u, "v": v}
    a, gen = _matrix(case, seed)
    x = _extra(case, gen)
    k, l, N = case["k"], case["k"] + case["p"], case["N"]
    out, a_sk, c_sk = {}, a, case
    if case["op"] == "train":
        om = x["omega"].to(_F64)
    else:
        om = _omega(int(seed) & 0x7FFFFFFF, case["n"], N * l)
        if case["dtype"] in ("f32", "bf16"):
            om = om.float().to(_STORED[case["dtype"]]).to(_F64)
        elif case["dtype"] == "fp8":
            om = om.float().to(torch.float8_e4m3fn).to(_F64)
            a_sk, scale = _dequantized(a, case["order"])
            c_sk = {**case, "order": "R"}
            out = {"codes": None, "scale": scale}
            a = a.to(torch.bfloat16)
    y = _mul(c_sk, a_sk, om)
    del om, a_sk
    qs = _bases(y, N)
    del y
    q = _hierarchical(qs, N) if case["integ"] == "HR" else _kolmogorov_nagumo(qs, N, l)
    del qs
    s, u, v = _triplets(case, a, q)
    uk, vk = _signed(u[:, :k], v[:, :k])
    if case["op"] != "train":
        return {**out, "s": s, "u": uk, "v": vk}
    u, v = torch.cat((uk, u[:, k:]), 1), torch.cat((vk, v[:, k:]), 1)
    for i in range(k, l):  # the other triplets keep the sign that the pair has together
        if float((_tmul(case, a, u[:, i:i + 1]) * v[:, i:i + 1]).sum()) < 0:
            v[:, i] = -v[:, i]
    da = _gradient(case, a, s, u, v, *(x[t].to(_F64) for t in ("gs", "gu", "gv")))
    return {"s": s[:k], "u": uk, "v": vk, "da": da}
