"""The one-launch triangular solves behind chol_solve_, ldlt solves and
qr_solve_: orders around a 16-row tile and a 128-row block, one to several
passes of 16 right-hand sides, both triangles, unaligned views, and the number
of right-hand sides at which the GEMM form takes over.

Bounds: a substitution's computed solution solves a system whose factor is
off by at most n·eps in every element (c = 4 for the 16×16 inverses and the
two solves), so ‖A x − b‖ ≤ 4 n eps ‖L‖_F² ‖x‖_F with A = L Lᵀ."""
import threading

import numpy as np
import pytest

from conftest import eps_of

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ORDERS = [1, 2, 15, 16, 17, 31, 113, 127, 128, 129, 144, 255, 256, 257, 400, 1025]


def _factor(n, rng, dtype, uplo, ld):
    """A triangular factor in a view with leading dimension ld, NaN elsewhere."""
    import gla

    L = np.tril(rng.standard_normal((n, n))) / np.sqrt(n)
    L[np.arange(n), np.arange(n)] = 1 + rng.random(n)
    L = L.astype(dtype)
    big = gla.empty_colmajor(ld, n, dtype=torch.float64 if dtype == np.float64 else torch.float32)
    big.fill_(float("nan"))
    F = big[1:1 + n, :]
    M = np.where(np.tri(n, dtype=bool), L, np.nan)
    F.copy_(torch.from_numpy(M if uplo == "L" else M.T.copy()))
    return L.astype(np.float64), F


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("n", ORDERS)
def test_cholesky_solve(n, uplo, dtype):
    import gla

    rng = np.random.default_rng(n)
    L, F = _factor(n, rng, dtype, uplo, n + 3)
    for nrhs in (1, 16, 17, 33):
        B = rng.standard_normal((n, nrhs)).astype(dtype)
        big = gla.empty_colmajor(n + 2, nrhs, dtype=F.dtype)
        big.fill_(3.0)
        X = big[1:1 + n, :]
        X.copy_(torch.from_numpy(B))
        gla.chol_solve_(F, X, uplo)
        x = gla.to_numpy(X).astype(np.float64)
        r = L @ (L.T @ x) - B
        assert np.linalg.norm(r) <= (4 * n * eps_of(dtype) * np.linalg.norm(L) ** 2 *
                                     np.linalg.norm(x))
        rest = gla.to_numpy(big)
        assert (rest[0] == 3).all() and (rest[1 + n] == 3).all()


@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("n", [1, 16, 100, 129, 257])
def test_ldlt_solve(n, uplo):
    """L D Lᵀ x = b, the unit diagonal not read from F (which holds D)."""
    import gla

    rng = np.random.default_rng(n)
    B0 = rng.standard_normal((n, n))
    A = B0 @ B0.T + n * np.eye(n)
    F = gla.ldlt(gla.Hermitian(gla.colmajor(A), uplo))
    for nrhs in (1, 20):
        B = rng.standard_normal((n, nrhs))
        X = gla.colmajor(B)
        F.ldiv_(X)
        x = gla.to_numpy(X)
        assert np.linalg.norm(A @ x - B) <= 20 * n * eps_of(np.float64) * np.linalg.norm(
            A) * np.linalg.norm(x)


@pytest.mark.parametrize("m,n,nrhs", [(1, 1, 1), (20, 16, 3), (130, 128, 17), (300, 129, 1),
                                      (700, 257, 33)])
def test_least_squares(m, n, nrhs):
    """The normal equations' residual: ‖Aᵀ(A x − b)‖ ≤ 20 m eps ‖A‖² (‖x‖ + ‖b‖)."""
    import gla

    rng = np.random.default_rng(m)
    A, B = rng.standard_normal((m, n)), rng.standard_normal((m, nrhs))
    F = gla.qrBlocked_(gla.colmajor(A), 12)
    X = gla.colmajor(B)
    x = gla.to_numpy(gla.qr_solve_(F, X))[:n]
    r = A.T @ (A @ x - B)
    a = np.linalg.norm(A)
    assert np.linalg.norm(r) <= 20 * m * eps_of(np.float64) * a * a * (
        np.linalg.norm(x) + np.linalg.norm(B))


@pytest.mark.parametrize("uplo", ["L", "U"])
def test_many_right_hand_sides(uplo):
    """The last count of the one form and the first of the other."""
    import gla

    n = 200
    rng = np.random.default_rng(7)
    L, F = _factor(n, rng, np.float64, uplo, n + 2)
    for nrhs in (2048, 2049):
        B = rng.standard_normal((n, nrhs))
        X = gla.colmajor(B)
        gla.chol_solve_(F, X, uplo)
        x = gla.to_numpy(X)
        assert np.linalg.norm(L @ (L.T @ x) - B) <= (4 * n * eps_of(np.float64) *
                                                     np.linalg.norm(L) ** 2 * np.linalg.norm(x))


def test_captured_solve_replays():
    import gla

    n, nrhs = 700, 20
    rng = np.random.default_rng(1)
    L, F = _factor(n, rng, np.float64, "L", n + 2)
    B = [gla.colmajor(rng.standard_normal((n, nrhs))) for _ in range(3)]
    ref = [gla.chol_solve_(F, b.clone(), "L") for b in B]
    X = B[0].clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        gla.chol_solve_(F, X, "L")
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gla.chol_solve_(F, X, "L")
    for b, r in zip(B, ref):
        X.copy_(b)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(X, r)


def test_solves_on_several_streams_at_once():
    """Four threads, each with a handle and a stream of its own and more
    workgroups than the device holds at once between them."""
    import ctypes as C

    import gla

    n, nrhs = 2500, 400
    lib = gla.lib()
    rng = np.random.default_rng(2)
    L, F = _factor(n, rng, np.float64, "L", n + 2)
    B = gla.colmajor(rng.standard_normal((n, nrhs)))
    ref = gla.chol_solve_(F, B.clone(), "L")
    torch.cuda.synchronize()
    bad = []

    def work():
        h = C.c_void_p()
        assert lib.gla_handle_create(C.byref(h)) == 0
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(3):
                X = B.clone()
                rc = lib.gla_chol_solve_d(h, b"L", n, nrhs, C.c_void_p(F.data_ptr()), n + 2,
                                          C.c_void_p(X.data_ptr()), n, C.c_void_p(s.cuda_stream))
                s.synchronize()
                if rc != 0 or not torch.equal(X, ref):
                    bad.append(rc)
        assert lib.gla_handle_destroy(h) == 0

    ts = [threading.Thread(target=work) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_wait_gives_up():
    import gla

    n = 2000
    rng = np.random.default_rng(3)
    L, F = _factor(n, rng, np.float64, "L", n + 2)
    B = gla.colmajor(rng.standard_normal((n, 1)))
    with gla.tuning(spin_limit=1):
        X = gla.chol_solve_(F, B.clone(), "L")
        torch.cuda.synchronize()
        assert not torch.isfinite(X).all()
    assert torch.isfinite(gla.chol_solve_(F, B.clone(), "L")).all()
