"""The work that a program using this package has it do, as cases to be timed.

Each listed case is one call (or one call and the solve that follows it) as a
user's program makes it, over the families the package holds: Cholesky factors
and solves, Householder QR and least squares, mixed precision with refinement,
uneven batches, the batched adjoint, the two-sided reductions that eigenvalues
and singular values start from, and complex QR.  The factorisations work in
place, so a pass copies its matrix first, as cholRecursive!(copy(A)) does.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "genericlinearalgebra.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import gla  # noqa: E402

_DT = {"f32": torch.float32, "f64": torch.float64, "c128": torch.complex128}


def listed():
    return [
        # a small covariance or normal-equations matrix: launches and the
        # pivot check are the whole call
        {"name": "chol_f64_100", "op": "chol", "dtype": "f64", "n": 100, "uplo": "L"},
        # the size the reference quotes its own Cholesky time on
        {"name": "chol_f64_1000", "op": "chol", "dtype": "f64", "n": 1000, "uplo": "L"},
        # the benchmark's large Cholesky
        {"name": "chol_f64_16384", "op": "chol", "dtype": "f64", "n": 16384, "uplo": "L"},
        # a kernel or Gaussian-process solve in single precision at an odd
        # size, upper factor, a block of right-hand sides
        {"name": "posv_f32_5001", "op": "posv", "dtype": "f32", "n": 5001, "nrhs": 16,
         "uplo": "U"},
        # the benchmark's blocked QR
        {"name": "qr_f64_8192x4096", "op": "qr", "dtype": "f64", "m": 8192, "n": 4096,
         "block": 128},
        # an ordinary regression: ragged shape, the default block size, one
        # right-hand side
        {"name": "lsq_f64_1501x700", "op": "lsq", "dtype": "f64", "m": 1501, "n": 700,
         "block": 12, "nrhs": 1},
        # mixed-precision solve with refinement to 1e-12, 16 right-hand sides
        {"name": "mixed_8192", "op": "mixed", "n": 8192, "nrhs": 16, "kappa": 1e2},
        # the benchmark's uneven batch: factor and solve, one right-hand side
        {"name": "batched_f64_10000", "op": "batched", "dtype": "f64", "count": 10000,
         "lo": 8, "hi": 256},
        # the backward pass of a layer that factors a batch of covariances
        {"name": "chol_grad_f64_512x128", "op": "chol_grad", "dtype": "f64", "count": 512,
         "n": 128},
        # what eigvals of a covariance matrix (principal components) starts with
        {"name": "symtri_f64_2048", "op": "symtri", "n": 2048, "uplo": "L"},
        # what svdvals of a tall matrix starts with
        {"name": "bidiag_f64_2500x1501", "op": "bidiag", "m": 2500, "n": 1501},
        # complex QR (steering matrices, impedance and scattering problems)
        {"name": "qr_c128_4096x2048", "op": "qr", "dtype": "c128", "m": 4096, "n": 2048,
         "block": 32},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["chol", "posv", "qr", "lsq", "mixed", "batched", "chol_grad", "symtri",
                     "bidiag", "zqr"])
    real = rng.choice(["f64", "f64", "f32"])
    uplo = rng.choice(["L", "L", "U"])
    if op == "chol":
        return {"op": op, "dtype": real, "n": _log(rng, 50, 12000), "uplo": uplo}
    if op == "posv":
        return {"op": op, "dtype": real, "n": _log(rng, 50, 6000),
                "nrhs": rng.choice([1, 3, 16, 40]), "uplo": uplo}
    if op in ("qr", "zqr"):
        n = _log(rng, 40, 3000 if op == "qr" else 1600)
        return {"op": "qr", "dtype": "f64" if op == "qr" else "c128",
                "m": n + _log(rng, 1, 5000 if op == "qr" else 2500), "n": n,
                "block": rng.choice([12, 32, 64, 128])}
    if op == "lsq":
        n = _log(rng, 20, 1200)
        return {"op": op, "dtype": real, "m": n + _log(rng, n, 4000), "n": n,
                "block": rng.choice([12, 32, 64, 128]), "nrhs": rng.choice([1, 4, 16])}
    if op == "mixed":
        return {"op": op, "n": _log(rng, 300, 8192), "nrhs": rng.choice([1, 8, 16]),
                "kappa": rng.choice([10.0, 30.0, 100.0])}
    if op == "batched":
        return {"op": op, "dtype": real, "count": _log(rng, 100, 10000), "lo": rng.randint(1, 16),
                "hi": rng.randint(32, 256)}
    if op == "chol_grad":
        return {"op": op, "dtype": real, "count": _log(rng, 16, 1000), "n": rng.randint(5, 128)}
    if op == "symtri":
        return {"op": op, "n": _log(rng, 64, 2300), "uplo": uplo}
    n = _log(rng, 64, 1600)
    return {"op": op, "m": n + _log(rng, 1, 1200), "n": n}


# ------------------------------------------------------------------ inputs --
def _randn(g, *shape, dtype=torch.float64):
    """N(0,1) in column-major order for matrices."""
    if len(shape) == 2:
        return _randn(g, shape[0] * shape[1], dtype=dtype).view(shape[1], shape[0]).t()
    if dtype.is_complex:
        return torch.complex(torch.randn(*shape, dtype=torch.float64, device="cuda", generator=g),
                             torch.randn(*shape, dtype=torch.float64, device="cuda", generator=g))
    return torch.randn(*shape, dtype=dtype, device="cuda", generator=g)


def _spd(g, n, dtype):
    """BᵀB + n·I with B iid N(0,1), formed in 64 bits."""
    B = _randn(g, n, n)
    A = B.t() @ B
    del B
    A.diagonal().add_(n)
    return _colmajor((0.5 * (A + A.t())).to(dtype))


def _colmajor(A):
    return A.t().contiguous().t()


def _spectrum(g, n, kappa):
    """Q diag(σ) Qᵀ, σ log-spaced over [1/κ, 1], Q a random orthogonal matrix
    (random signs between two orthonormal sine transforms)."""
    k = torch.arange(1, n + 1, device="cuda")
    S = torch.outer(k, k).remainder_(2 * (n + 1)).to(torch.float64)
    S = S.mul_(math.pi / (n + 1)).sin_().mul_(math.sqrt(2.0 / (n + 1)))
    s1, s2 = (torch.randn(n, dtype=torch.float64, device="cuda", generator=g).sign()
              for _ in range(2))
    Q = s1[:, None] * (S @ (s2[:, None] * S))
    del S
    A = (Q * torch.logspace(0, -math.log10(kappa), n, dtype=torch.float64, device="cuda")) @ Q.t()
    return _colmajor(0.5 * (A + A.t()))


def _sizes(case):
    rng = np.random.default_rng(case["count"])
    return rng.integers(case["lo"], case["hi"] + 1, size=case["count"])


def _groups(sizes):
    """For each order n of the batch: n, the matrices' indices, their places
    in the packed A and b (one row per matrix)."""
    aoff = np.concatenate([[0], np.cumsum(sizes * sizes)])
    boff = np.concatenate([[0], np.cumsum(sizes)])
    for n in np.unique(sizes):
        i = np.nonzero(sizes == n)[0]
        ai = torch.from_numpy(aoff[i]).cuda()[:, None] + torch.arange(n * n, device="cuda")
        bi = torch.from_numpy(boff[i]).cuda()[:, None] + torch.arange(n, device="cuda")
        yield int(n), i, ai, bi


def _spd_batch(g, count, n, dtype):
    B = _randn(g, count, n, n)
    A = torch.bmm(B.transpose(1, 2).contiguous(), B)
    A.diagonal(dim1=1, dim2=2).add_(n)
    return (0.5 * (A + A.transpose(1, 2))).to(dtype).contiguous()


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, dt = case["op"], _DT[case.get("dtype", "f64")]
    if op == "chol":
        return {"A": _spd(g, case["n"], dt)}
    if op == "posv":
        return {"A": _spd(g, case["n"], dt), "B": _randn(g, case["n"], case["nrhs"], dtype=dt)}
    if op in ("qr", "lsq", "bidiag"):
        s = {"A": _randn(g, case["m"], case["n"], dtype=dt)}
        if op == "lsq":
            s["B"] = _randn(g, case["m"], case["nrhs"], dtype=dt)
        return s
    if op == "mixed":
        return {"A": _spectrum(g, case["n"], case["kappa"]),
                "B": _randn(g, case["n"], case["nrhs"])}
    if op == "symtri":
        return {"A": _spd(g, case["n"], dt)}
    if op == "chol_grad":
        # (batch, n, n), each matrix column-major
        return {"A": _spd_batch(g, case["count"], case["n"], dt).transpose(1, 2),
                "W": _randn(g, case["count"], case["n"], case["n"], dtype=dt).transpose(1, 2)}
    sizes = _sizes(case)
    A = torch.zeros(int((sizes * sizes).sum()) + 1, dtype=dt, device="cuda")
    b = torch.zeros(int(sizes.sum()) + 1, dtype=dt, device="cuda")
    for n, i, ai, bi in _groups(sizes):
        A[ai] = _spd_batch(g, len(i), n, dt).view(len(i), n * n)
        b[bi] = _randn(g, len(i), n, dtype=dt)
    return {"sizes": sizes, "A": A, "b": b}


def prepare(case, seed):
    """Inputs on the GPU, the buffers a program that factors in a loop keeps,
    and for a batch its plan and packed storage."""
    s = dict(_inputs(case, seed), case=case)
    op = case["op"]
    if op == "batched":
        s["packed"] = gla.PackedBatch(s["sizes"], s["A"].dtype)
        s["plan"] = gla.BatchPlan(s["sizes"], s["A"].dtype)
    elif op == "chol_grad":
        s["out"] = torch.empty_like(s["A"])
    elif op != "mixed":
        s["W"] = torch.empty_like(s["A"])
        if "B" in s:
            s["X"] = torch.empty_like(s["B"])
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ a pass --
def run(s):
    case = s["case"]
    op = case["op"]
    if op == "mixed":
        X, _ = gla.chol_solve_mixed(s["A"], s["B"], precision="auto", tol=1e-12)
        return X
    if op == "batched":
        pb = s["packed"]
        pb.A.copy_(s["A"])
        pb.b.copy_(s["b"])
        gla.chol_solve_batched_(s["plan"], pb.A_ptrs, pb.lda, pb.b_ptrs, pb.info)
        return {"A": pb.A, "b": pb.b, "info": pb.info}
    if op == "chol_grad":
        return gla.chol_adjoint_batched(s["A"], s["W"], "S", out=s["out"])
    W = s["W"]
    W.copy_(s["A"])
    if op == "chol":
        return gla.cholRecursive_(W, case["uplo"]).data
    if op == "posv":
        F = gla.cholRecursive_(W, case["uplo"])
        s["X"].copy_(s["B"])
        return {"X": gla.chol_solve_(F, s["X"]), "F": F.data}
    if op == "qr":
        F = gla.qrBlocked_(W, case["block"])
        return {"factors": F.factors, "tau": F.tau}
    if op == "lsq":
        F = gla.qrBlocked_(W, case["block"])
        s["X"].copy_(s["B"])
        x = gla.qr_solve_(F, s["X"])
        return {"x": x, "factors": F.factors, "tau": F.tau}
    if op == "symtri":
        F = gla.symtri_(gla.Hermitian(W, case["uplo"]))
        d, e = F.diagonals
        return {"factors": F.factors, "tau": F.tau, "d": d, "e": e}
    F = gla.bidiagonalize_(W)
    d, e = F.bidiagonal
    return {"factors": F.factors, "taul": F.taul, "taur": F.taur, "d": d, "e": e}


# -------------------------------------------------------------- least work --
def work(case):
    op = case["op"]
    z = 4 if case.get("dtype") == "f32" else 16 if case.get("dtype") == "c128" else 8
    c = 4 if case.get("dtype") == "c128" else 1
    if op == "batched":
        n = _sizes(case).astype(np.float64)
        return {"bytes": float(np.sum(z * (n * (n + 1) + 2 * n))),
                "flops": float(np.sum(n ** 3 / 3 + 2 * n ** 2))}
    n = float(case["n"])
    if op == "chol":
        return {"bytes": z * n * (n + 1), "flops": n ** 3 / 3}
    if op == "posv":
        r = case["nrhs"]
        return {"bytes": z * (n * (n + 1) + 2 * n * r), "flops": n ** 3 / 3 + 2 * n * n * r}
    if op == "mixed":
        # the lower triangle in, the solution out; the factor stays inside
        r = case["nrhs"]
        return {"bytes": z * (n * (n + 1) / 2 + 2 * n * r), "flops": n ** 3 / 3 + 2 * n * n * r}
    if op == "chol_grad":
        # factor (n³/3) and adjoint (7n³/3); two triangles in, one matrix out
        k = case["count"]
        return {"bytes": z * k * (n * (n + 1) + n * n), "flops": k * 8 * n ** 3 / 3}
    if op == "symtri":
        return {"bytes": z * n * (n + 1), "flops": 4 * n ** 3 / 3}
    m = float(case["m"])
    if op == "bidiag":
        return {"bytes": 2 * z * m * n, "flops": 4 * m * n * n - 4 * n ** 3 / 3}
    f = c * (2 * m * n * n - 2 * n ** 3 / 3)
    if op == "lsq":
        r = case["nrhs"]
        return {"bytes": z * (2 * m * n + (m + n) * r), "flops": f + r * (4 * m * n - n * n)}
    return {"bytes": 2 * z * m * n, "flops": f}


# ------------------------------------------------------- values in 64 bits --
def _reflect(x):
    """reflector!: the stored column (−ν, v₂, …), v with v₁ = 1, and τ."""
    nu = torch.copysign(torch.linalg.vector_norm(x), x[0])
    xi = x[0] + nu
    v = x / xi
    v[0] = 1
    out = v.clone()
    out[0] = -nu
    return out, v, xi / nu


def _symtri_lower(A):
    n = A.shape[0]
    S, F = A.clone(), A.clone()
    tau = torch.zeros(max(n - 1, 0), dtype=A.dtype, device=A.device)
    for k in range(n - 2):
        F[k:, k] = S[k:, k]
        F[k + 1:, k], v, t = _reflect(S[k + 1:, k])
        tau[k] = t
        T = S[k + 1:, k + 1:]
        p = t * (T @ v)
        w = p - (t / 2 * (v @ p)) * v
        T.addr_(v, w, alpha=-1).addr_(w, v, alpha=-1)
    F[n - 2:, n - 2:] = torch.tril(S[n - 2:, n - 2:]) + torch.triu(A[n - 2:, n - 2:], 1)
    return F, tau


def _bidiag(A):
    m, n = A.shape
    F = A.clone()
    tl = torch.zeros(n, dtype=A.dtype, device=A.device)
    tr = torch.zeros(max(n - 1, 0), dtype=A.dtype, device=A.device)
    for i in range(n):
        F[i:, i], v, tl[i] = _reflect(F[i:, i].clone())
        if i + 1 < n:
            T = F[i:, i + 1:]
            T.addr_(v, tl[i] * (v @ T), alpha=-1)
            F[i, i + 1:], v, tr[i] = _reflect(F[i, i + 1:].clone())
            T = F[i + 1:, i + 1:]
            T.addr_(tr[i] * (T @ v), v, alpha=-1)
    return F, tl, tr


def exact(case, seed):
    """What run returns, by torch in 64 bits.  The factorisations are unique:
    L with a positive diagonal, reflectors with the sign that reflector! and
    LAPACK take."""
    op = case["op"]
    s = _inputs(case, seed)
    if op == "batched":
        A, b = s["A"].double(), s["b"].double()
        for n, i, ai, bi in _groups(s["sizes"]):
            M = A[ai].view(len(i), n, n)
            L = torch.linalg.cholesky(M)
            b[bi] = torch.cholesky_solve(b[bi][:, :, None], L)[:, :, 0]
            # packed by columns: row c of the view is column c of the matrix
            A[ai] = (L.transpose(1, 2) + torch.tril(M, -1)).reshape(len(i), n * n)
        return {"A": A, "b": b, "info": torch.zeros(case["count"], dtype=torch.int32)}
    A = s["A"].to(torch.complex128 if s["A"].is_complex() else torch.float64)
    if op == "chol_grad":
        L = torch.linalg.cholesky(A.cpu())
        W = torch.tril(s["W"].double().cpu())
        P = torch.tril(torch.bmm(L.transpose(1, 2).contiguous(), W))
        P.diagonal(dim1=1, dim2=2).mul_(0.5)
        Y = torch.linalg.solve_triangular(L.transpose(1, 2).contiguous(), P + P.transpose(1, 2),
                                          upper=True)
        return 0.5 * torch.linalg.solve_triangular(L, Y, upper=False, left=False)
    if op == "mixed":
        return torch.cholesky_solve(s["B"], torch.linalg.cholesky(A))
    if op in ("chol", "posv"):
        L = torch.linalg.cholesky(A)
        F = torch.tril(L) + torch.triu(A, 1) if case["uplo"] == "L" else L.t() + torch.tril(A, -1)
        if op == "chol":
            return F
        return {"X": torch.cholesky_solve(s["B"].double(), L), "F": F}
    if op in ("qr", "lsq"):
        F, tau = torch.geqrf(A)
        if op == "qr":
            return {"factors": F, "tau": tau}
        n = case["n"]
        y = torch.ormqr(F, tau, s["B"].double(), left=True, transpose=True)[:n]
        x = torch.linalg.solve_triangular(torch.triu(F[:n]), y, upper=True)
        return {"x": x, "factors": F, "tau": tau}
    if op == "symtri":
        if case["uplo"] == "L":
            F, tau = _symtri_lower(A)
            return {"factors": F, "tau": tau, "d": F.diagonal(), "e": F.diagonal(-1)}
        F, tau = _symtri_lower(A.flip(0, 1))
        F = F.flip(0, 1)
        return {"factors": F, "tau": tau, "d": F.diagonal(), "e": F.diagonal(1)}
    F, tl, tr = _bidiag(A)
    return {"factors": F, "taul": tl, "taur": tr, "d": F.diagonal(), "e": F.diagonal(1)}


if __name__ == "__main__":
    for c in listed() + [draw(random.Random(i)) for i in range(4)]:
        print(c, work(c))
