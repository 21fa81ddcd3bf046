"""Performance cases of slepc_amd: the calls a program that computes eigenpairs
with this package spends its time in, each through the public entry points.

The kinds, by what they stand for in real use:

  ortho    BV.copy_column + BV.orthonormalize_column: one vector against a basis
           (start vectors, locking, programs that drive the basis themselves);
           the smallest call, where launches and latency count.
  spmv     Mat.mult: the operator on its own.
  sweep    BV.mat_arnoldi: the Arnoldi / Lanczos expansion, where a Krylov-Schur
           solve spends nearly all of its time (k = 0: the first sweep, k > 0:
           the sweep after a restart that kept k columns).
  restart  BV.multinplace: the basis update of a restart.
  project  BV.matmult + BV.dot: Y = A X and M = Y^T X, a Rayleigh-Ritz projection.
  orth     BV.orthogonalize: a block made orthonormal (Cholesky QR or TSQR).
  solve    EPS: a whole Krylov-Schur solve with its eigenvectors.
  batch    Batch: many uneven symmetric problems solved together.

Operators: 5-point Laplacians (lap2d), the finite-volume diffusion family
(fv2d), 3-D convection-diffusion (convdiff3d, non-symmetric) and the 27-point
stencil with a random diagonal (stencil27), in FP64 and in the FP32 that the
first phase of a mixed-precision solve runs in.
"""
import math

import numpy as np
import torch

import slepc_amd as sa
from slepc_amd.batch import Batch

FP32_TOL_STEPS = 48      # longest FP32 sweep that the ranges hold


def listed():
    return [
        # one vector against 20 columns of a 100 x 100 grid's basis
        dict(name="ortho_n10000_j20", kind="ortho", n=10000, j=20, prec="fp64"),
        # the operator of the 256 x 256 diffusion family: a cache-resident SpMV
        dict(name="spmv_fv2d_256", kind="spmv", op="fv2d", nx=256, ny=256, nz=1, prec="fp64"),
        # the 27-point operator at 128^3: an SpMV streamed from HBM
        dict(name="spmv_stencil27_128", kind="spmv", op="stencil27", nx=128, ny=128, nz=128, prec="fp64"),
        # 100 x 100 Laplacian, ncv 32: a restart's sweep of a small problem
        dict(name="sweep_lap2d_100", kind="sweep", op="lap2d", nx=100, ny=100, nz=1, k=16, m=32, prec="fp64"),
        # the 256 x 256 diffusion family, ncv 64: its first sweep
        dict(name="sweep_fv2d_256", kind="sweep", op="fv2d", nx=256, ny=256, nz=1, k=0, m=64, prec="fp64"),
        # convection-diffusion at 128^3, ncv 64: a restart's sweep of a large problem
        dict(name="sweep_convdiff_128", kind="sweep", op="convdiff3d", nx=128, ny=128, nz=128, k=32, m=64,
             prec="fp64"),
        # 27-point operator on an odd grid, ncv 96, in FP32 (first phase of a mixed solve)
        dict(name="sweep_stencil27_f32", kind="sweep", op="stencil27", nx=121, ny=113, nz=97, k=48, m=96,
             prec="fp32"),
        # restart of ncv 96 keeping 48 at 128^3
        dict(name="restart_128_K96_N48", kind="restart", n=2097152, K=96, N=48, prec="fp64"),
        # projection onto 32 columns at 128^3
        dict(name="project_convdiff_128", kind="project", op="convdiff3d", nx=128, ny=128, nz=128, nc=32,
             prec="fp64"),
        # tall-skinny QR of 32 columns at 128^3
        dict(name="tsqr_128_k32", kind="orth", n=2097152, nc=32, method="tsqr", prec="fp64"),
        # six largest eigenpairs of a rectangular Laplacian, whole solve
        dict(name="solve_lap2d_100x70", kind="solve", nx=100, ny=70, nev=6, ncv=24, tol=1e-10),
        # 24 uneven Laplacians with a random potential solved together
        dict(name="batch_24", kind="batch", P=24, lo=32, hi=160, nev=8, ncv=24, tol=1e-10),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, op, lo, hi):
    """A grid of about lo..hi rows (log-uniform), sides uneven."""
    n = _logint(rng, lo, hi)
    if op in ("lap2d", "fv2d"):
        nx = max(8, int(math.sqrt(n) * rng.uniform(0.7, 1.4)))
        return nx, max(8, n // nx), 1
    a = n ** (1.0 / 3.0)
    nx, ny = max(6, int(a * rng.uniform(0.8, 1.25))), max(6, int(a * rng.uniform(0.8, 1.25)))
    return nx, ny, max(6, n // (nx * ny))


def draw(rng):
    kind = rng.choice(["ortho", "spmv", "sweep", "sweep", "sweep", "restart", "project", "orth", "solve", "batch"])
    prec = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "ortho":
        return dict(kind=kind, n=_logint(rng, 2000, 1500000), j=rng.randint(1, 95), prec=prec)
    if kind == "spmv":
        op = rng.choice(["lap2d", "fv2d", "convdiff3d", "stencil27"])
        nx, ny, nz = _grid(rng, op, 3000, 2000000)
        return dict(kind=kind, op=op, nx=nx, ny=ny, nz=nz, prec=prec)
    if kind == "sweep":
        op = rng.choice(["lap2d", "fv2d", "convdiff3d", "stencil27"])
        m = rng.randint(16, 96)
        k = rng.choice([0, m // 2])
        if prec == "fp32":
            k = max(k, m - FP32_TOL_STEPS)
        nx, ny, nz = _grid(rng, op, 2000, 1000000)
        return dict(kind=kind, op=op, nx=nx, ny=ny, nz=nz, k=k, m=m, prec=prec)
    if kind == "restart":
        K = rng.randint(16, 96)
        return dict(kind=kind, n=_logint(rng, 5000, 2000000), K=K, N=max(4, int(K * rng.uniform(0.4, 0.7))), prec=prec)
    if kind == "project":
        op = rng.choice(["lap2d", "convdiff3d", "stencil27"])
        nx, ny, nz = _grid(rng, op, 5000, 1500000)
        return dict(kind=kind, op=op, nx=nx, ny=ny, nz=nz, nc=rng.randint(4, 40), prec=prec)
    if kind == "orth":
        return dict(kind=kind, n=_logint(rng, 5000, 1500000), nc=rng.randint(4, 48),
                    method=rng.choice(["tsqr", "tsqr", "chol"]), prec=prec)
    if kind == "solve":
        nx = rng.randint(60, 150)
        return dict(kind=kind, nx=nx, ny=int(nx * rng.uniform(0.69, 0.72)), nev=rng.randint(3, 6),
                    ncv=rng.randint(20, 32), tol=1e-10)
    return dict(kind=kind, P=rng.randint(8, 24), lo=32, hi=rng.randint(96, 160), nev=8, ncv=24, tol=1e-10)


# ---------------------------------------------------------------- helpers
def _prec(case):
    return sa.FP64 if case.get("prec", "fp64") == "fp64" else sa.FP32


def _dtype(case):
    return torch.float64 if case.get("prec", "fp64") == "fp64" else torch.float32


def _operator(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["op"] == "lap2d":
        return sa.lap2d(nx, ny)
    if case["op"] == "fv2d":
        return sa.fv2d(nx, ny, sa.fv_theta(5, seed % 100000))
    if case["op"] == "convdiff3d":
        return sa.convdiff3d(nx, ny, nz)
    return sa.stencil27(nx, ny, nz, seed=1 + seed % 100000)


def _rows(case):
    return case["nx"] * case["ny"] * case["nz"] if "nx" in case else case["n"]


def _nnz(case):
    """Nonzeros of the operator (2-D: 5-point, 3-D: 7 or 27 points)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["op"] in ("lap2d", "fv2d"):
        return 5 * nx * ny - 2 * nx - 2 * ny
    if case["op"] == "convdiff3d":
        return 7 * nx * ny * nz - 2 * (nx * ny + ny * nz + nx * nz)
    return (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)


class _Columns:
    """The device memory of a basis, for torch to look at."""

    def __init__(self, V, ncols):
        f4 = V.prec == sa.FP32
        self.keep = V
        self.__cuda_array_interface__ = dict(shape=(ncols, V.ld), typestr="<f4" if f4 else "<f8",
                                             data=(V.column_ptr(0).value, False), version=3, strides=None)


def _view(V, ncols):
    """ncols x n tensor over the basis: row j is column j."""
    return torch.as_tensor(_Columns(V, ncols), device="cuda")[:, :V.n]


def _rand(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64) * 2.0 - 1.0


def _orthonormal_rows(seed, k, n):
    """k orthonormal rows of length n (Cholesky QR twice on random rows)."""
    X = _rand(seed, k, n)
    for _ in range(2):
        L = torch.linalg.cholesky(X @ X.T)
        X = torch.linalg.inv(L) @ X
    return X


def _block(seed, nc, n):
    """nc rows of length n, each leaning on the one before it."""
    X = _rand(seed, nc, n)
    X[1:] += 0.8 * X[:-1].clone()
    return X


def _coefficients(case, seed):
    """Orthonormal K x N restart coefficients."""
    A = np.random.default_rng(seed).standard_normal((case["K"], case["N"]))
    return np.linalg.qr(A)[0]


def _start(seed, n):
    return np.random.default_rng(seed).uniform(-1.0, 1.0, n)


def _batch_sides(case):
    """The grid sides of the batch's problems: the case's own, whatever the seed."""
    rng = np.random.default_rng([case["P"], case["lo"], case["hi"]])
    return [(int(a), int(b)) for a, b in rng.integers(case["lo"], case["hi"] + 1, (case["P"], 2))]


def _batch_csrs(case, seed):
    rng = np.random.default_rng(seed)
    return [sa.lap2d(nx, ny, 10.0, int(rng.integers(1, 1 << 30))) for nx, ny in _batch_sides(case)]


# ---------------------------------------------------------------- prepare / run
def prepare(case, seed):
    sa.init(0)
    kind, prec = case["kind"], _prec(case)
    s = dict(case=case)
    if kind == "ortho":
        j = case["j"]
        V = s["V"] = sa.BV(case["n"], j + 2, prec)
        view = s["view"] = _view(V, j + 2)
        view[:j] = _orthonormal_rows(seed, j, case["n"]).to(view.dtype)
        view[j + 1] = _rand(seed + 7919, case["n"]).to(view.dtype)
    elif kind == "spmv":
        s["A"] = sa.Mat(_operator(case, seed), prec)
        s["x"] = _rand(seed, _rows(case)).to(_dtype(case))
        s["y"] = torch.empty_like(s["x"])
    elif kind == "sweep":
        s["A"] = sa.Mat(_operator(case, seed), prec)
        V = s["V"] = sa.BV(_rows(case), case["m"] + 1, prec)
        view = s["view"] = _view(V, case["m"] + 1)
        view[:case["k"] + 1] = _orthonormal_rows(seed, case["k"] + 1, V.n).to(view.dtype)
    elif kind == "restart":
        V = s["V"] = sa.BV(case["n"], case["K"] + 1, prec)
        V.set_active_columns(0, case["K"])
        view = s["view"] = _view(V, case["K"] + 1)
        view[:case["K"]] = _rand(seed, case["K"], case["n"]).to(view.dtype)
        s["Q"] = np.zeros((case["K"], case["K"]))
        s["Q"][:, :case["N"]] = _coefficients(case, seed)
    elif kind == "project":
        s["A"] = sa.Mat(_operator(case, seed), prec)
        s["X"], s["Y"] = sa.BV(_rows(case), case["nc"], prec), sa.BV(_rows(case), case["nc"], prec)
        s["xview"], s["yview"] = _view(s["X"], case["nc"]), _view(s["Y"], case["nc"])
        s["xview"][:] = _block(seed, case["nc"], _rows(case)).to(s["xview"].dtype)
    elif kind == "orth":
        V = s["V"] = sa.BV(case["n"], case["nc"], prec)
        view = s["view"] = _view(V, case["nc"])
        view[:] = _block(seed, case["nc"], case["n"]).to(view.dtype)
    elif kind == "solve":
        s["A"] = sa.Mat(sa.lap2d(case["nx"], case["ny"]))
        s["v0"] = _start(seed, case["nx"] * case["ny"])
    else:
        csrs = _batch_csrs(case, seed)
        s["v0"] = [_start(seed + 1 + p, A.n) for p, A in enumerate(csrs)]
        s["B"] = Batch(csrs)
        s["B"].set_true_residual(True)
    torch.cuda.synchronize()      # the library works on a stream of its own
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ortho":
        V, j = state["V"], case["j"]
        V.copy_column(j + 1, j)
        norm, _ = V.orthonormalize_column(j)
        return dict(v=state["view"][j], norm=norm, h=V.coefficients(j, j + 1))
    if kind == "spmv":
        state["A"].mult(state["x"].data_ptr(), state["y"].data_ptr())
        return state["y"]
    if kind == "sweep":
        V, k, m = state["V"], case["k"], case["m"]
        steps, beta, _ = V.mat_arnoldi(state["A"], k, m)
        return dict(steps=steps, beta=beta, V=state["view"][k + 1:m + 1], H=V.coefficients(k + 1, m + 1))
    if kind == "restart":
        state["V"].multinplace(state["Q"], 0, case["N"])
        return state["view"][:case["N"]]
    if kind == "project":
        state["X"].matmult(state["A"], state["Y"])
        return dict(Y=state["yview"], M=state["X"].dot(state["Y"]))
    if kind == "orth":
        R = state["V"].orthogonalize(case["method"])
        return dict(Q=state["view"], R=R)
    if kind == "solve":
        E = sa.EPS()
        E.setOperators(state["A"])
        E.setProblemType(True)
        E.setWhichEigenpairs("LM")
        E.setDimensions(case["nev"], case["ncv"])
        E.setTolerances(case["tol"])
        E.setInitialSpace(state["v0"])
        E.solve()
        pairs = [E.getEigenpair(i) for i in range(case["nev"])]
        E.destroy()
        # an eigenvector's sign is free: each with a positive part along the start vector
        X = np.stack([p[2] * math.copysign(1.0, p[2] @ state["v0"]) for p in pairs])
        return dict(values=np.array([p[0] for p in pairs]), vectors=X)
    B, v0 = state["B"], state["v0"]
    B.solve(case["nev"], case["ncv"], case["tol"], "LM", v0=v0)
    values, vectors = [], []
    for p in range(case["P"]):
        pairs = [B.eigenpair(p, i) for i in range(case["nev"])]
        values.append([v for v, _ in pairs])
        vectors.append(np.stack([x * math.copysign(1.0, x @ v0[p]) for _, x in pairs]))
    return dict(values=np.array(values), vectors=np.concatenate([x.ravel() for x in vectors]))


# ---------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    es = 8 if case.get("prec", "fp64") == "fp64" else 4
    if kind == "ortho":
        n, j = case["n"], case["j"]
        return dict(bytes=(j + 2) * n * es, flops=8 * n * j)
    if kind in ("spmv", "sweep", "project"):
        n, nnz = _rows(case), _nnz(case)
        op = nnz * (es + 4) + 4 * (n + 1)
    if kind == "spmv":
        return dict(bytes=op + 2 * n * es, flops=2 * nnz)
    if kind == "sweep":
        # each step cannot start before the one before it has ended: it reads
        # the operator and the basis and writes its column; two passes of
        # classical Gram-Schmidt
        b = sum(op + (c + 1) * n * es for c in range(case["k"] + 1, case["m"] + 1))
        f = sum(2 * nnz + 8 * n * c for c in range(case["k"] + 1, case["m"] + 1))
        return dict(bytes=b, flops=f)
    if kind == "restart":
        n, K, N = case["n"], case["K"], case["N"]
        return dict(bytes=(K + N) * n * es, flops=2 * n * K * N)
    if kind == "project":
        nc = case["nc"]
        return dict(bytes=op + 2 * nc * n * es, flops=2 * nnz * nc + 2 * n * nc * nc)
    if kind == "orth":
        n, nc = case["n"], case["nc"]
        return dict(bytes=2 * nc * n * es, flops=4 * n * nc * nc)
    if kind == "solve":
        # at the least one basis is built: ncv steps
        n = case["nx"] * case["ny"]
        nnz = 5 * n - 2 * case["nx"] - 2 * case["ny"]
        return dict(bytes=case["ncv"] * (12 * nnz + 20 * n), flops=case["ncv"] * (2 * nnz + 4 * n * case["ncv"]))
    n = sum(nx * ny for nx, ny in _batch_sides(case))
    return dict(bytes=case["ncv"] * 80 * n, flops=case["ncv"] * (10 * n + 4 * n * case["ncv"]))


def tolerance(case):
    """About four times the largest error against 64-bit references measured over
    the ranges.  FP64: 2e-14 (sweeps of 96 steps, projections whose M cancels),
    FP32: 4e-6 (sweeps), 5e-7 (the rest).  A whole solve's eigenvectors are
    as exact as tol / gap makes them: 3e-8 for the Laplacian; the batch's
    random potentials leave closer eigenvalues than that."""
    kind, f32 = case["kind"], case.get("prec", "fp64") == "fp32"
    if kind == "solve":
        return dict(rel=5e-7, max=1e-5)
    if kind == "batch":
        return dict(rel=1e-4, max=0.02)
    if f32:
        return dict(rel=2e-5, max=5e-4) if kind == "sweep" else dict(rel=2e-6, max=1e-4)
    return dict(rel=1e-13, max=1e-10)


# ---------------------------------------------------------------- exact
def _ell(csr, dtype):
    """The operator as padded rows (columns, values in 64 bits of the stored precision) on the GPU."""
    n, rp = csr.n, csr.rowptr.astype(np.int64)
    w = int((rp[1:] - rp[:-1]).max())
    rows = torch.from_numpy(np.repeat(np.arange(n), rp[1:] - rp[:-1])).cuda()
    slot = torch.arange(len(csr.col), device="cuda") - torch.from_numpy(rp[:-1]).cuda()[rows]
    col = torch.zeros(w, n, dtype=torch.int64, device="cuda")
    val = torch.zeros(w, n, dtype=torch.float64, device="cuda")
    col[slot, rows] = torch.from_numpy(csr.col.astype(np.int64)).cuda()
    val[slot, rows] = torch.from_numpy(csr.val).cuda().to(dtype).double()
    return col, val


def _apply(ell, x):
    col, val = ell
    y = torch.zeros_like(x)
    for c, v in zip(col, val):
        y += v * x[c]
    return y


def _twice(V, v):
    """v orthonormalised against the rows of V by two passes: (v, coefficients, norm)."""
    h = V @ v
    v = v - V.T @ h
    g = V @ v
    v = v - V.T @ g
    norm = torch.linalg.vector_norm(v)
    return v / norm, h + g, float(norm)


def exact(case, seed):
    kind, dt = case["kind"], _dtype(case)
    if kind == "batch":
        return None
    if kind == "ortho":
        j, n = case["j"], case["n"]
        V = _orthonormal_rows(seed, j, n).to(dt).double()
        v, h, norm = _twice(V, _rand(seed + 7919, n).to(dt).double())
        H = np.zeros((j + 2, 1))
        H[:j, 0] = h.cpu().numpy()
        H[j, 0] = norm
        return dict(v=v, norm=norm, h=H)
    if kind == "spmv":
        return _apply(_ell(_operator(case, seed), dt), _rand(seed, _rows(case)).to(dt).double())
    if kind == "sweep":
        n, k, m = _rows(case), case["k"], case["m"]
        ell = _ell(_operator(case, seed), dt)
        V = torch.zeros(m + 1, n, dtype=torch.float64, device="cuda")
        V[:k + 1] = _orthonormal_rows(seed, k + 1, n).to(dt).double()
        H = np.zeros((m + 1, m - k))
        for c in range(k + 1, m + 1):
            V[c], h, norm = _twice(V[:c], _apply(ell, V[c - 1]))
            H[:c, c - k - 1] = h.cpu().numpy()
            H[c, c - k - 1] = norm
        return dict(steps=m, beta=float(norm), V=V[k + 1:], H=H)
    if kind == "restart":
        V = _rand(seed, case["K"], case["n"]).to(dt).double()
        return torch.from_numpy(_coefficients(case, seed)).cuda().T.contiguous() @ V
    if kind == "project":
        ell = _ell(_operator(case, seed), dt)
        X = _block(seed, case["nc"], _rows(case)).to(dt).double()
        Y = torch.stack([_apply(ell, x) for x in X])
        return dict(Y=Y, M=(Y @ X.T).cpu().numpy())
    if kind == "orth":
        X = _block(seed, case["nc"], case["n"]).to(dt).double().cpu()
        Q, R = torch.linalg.qr(X.T)
        sign = torch.sign(torch.diagonal(R)) if case["method"] == "chol" else torch.ones(case["nc"], dtype=R.dtype)
        return dict(Q=(Q * sign).T.contiguous(), R=(sign[:, None] * R).numpy())
    # the rectangular Laplacian's closed form
    nx, ny, nev = case["nx"], case["ny"], case["nev"]
    i, j = np.arange(1, nx + 1), np.arange(1, ny + 1)
    lam = 4.0 - 2.0 * np.cos(np.pi * i / (nx + 1))[None, :] - 2.0 * np.cos(np.pi * j / (ny + 1))[:, None]
    best = np.argsort(-lam, axis=None)[:nev]
    v0, X = _start(seed, nx * ny), []
    for b in best:
        q, p = divmod(int(b), nx)
        x = np.outer(np.sin(np.pi * (q + 1) * j / (ny + 1)), np.sin(np.pi * (p + 1) * i / (nx + 1))).ravel()
        X.append(x / np.linalg.norm(x) * math.copysign(1.0, x @ v0))
    return dict(values=lam.ravel()[best], vectors=np.stack(X))
