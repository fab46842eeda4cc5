"""symtri! with the matrix held in registers (orders up to 2048, and the last
2048 of larger ones): orders around a workgroup's eight rows and around the
limit, both triangles, against the same call under stream capture, which takes
the launch-per-column kernels, and the oracle; several streams at once, which
must follow one another; and a wait that gives up."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cov(n, rng, dtype=np.float64):
    B = rng.standard_normal((n, n))
    A = B.T @ B + n * np.eye(n)
    return ((A + A.T) / 2).astype(dtype)


@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("n", [3, 7, 8, 9, 15, 17, 63, 65, 255, 257, 264])
def test_orders_vs_oracle(n, uplo):
    import gla

    A = _cov(n, np.random.default_rng(n))
    big = gla.empty_colmajor(n + 5, n)
    X = big[3:3 + n, :]
    X.copy_(torch.from_numpy(A))
    F = gla.symtri_(gla.Hermitian(X, uplo))
    got, tau = gla.to_numpy(F.factors), F.tau.cpu().numpy()
    ref, tref = O.symtri(A, uplo)
    tru, ttru = O.symtri_quad(A, uplo)
    tri, other, k = (np.tril, np.triu, 1) if uplo == "L" else (np.triu, np.tril, -1)
    tol = 10 * n * eps_of(np.float64)
    assert rel(tri(got), tri(tru)) <= max(tol, 2 * rel(tri(ref), tri(tru)))
    assert rel(tau, ttru) <= max(tol, 2 * rel(tref, ttru))
    assert np.array_equal(other(got, k), other(A, k))


@pytest.mark.parametrize("n", [2047, 2048, 2049, 2100])
def test_at_the_limit(n):
    """Tridiagonal with the eigenvalues of A."""
    import gla
    import scipy.linalg as sl

    A = _cov(n, np.random.default_rng(n))
    F = gla.symtri_(gla.Hermitian(gla.colmajor(A), "L"))
    d, e = (x.cpu().numpy() for x in F.diagonals)
    la = np.linalg.eigvalsh(A)
    lt = sl.eigvalsh_tridiagonal(d, e)
    assert np.max(np.abs(lt - la)) <= 10 * n * eps_of(np.float64) * np.max(np.abs(la))


def test_captured_call_takes_the_launches():
    """Under capture the launch-per-column kernels run: the same reduction to
    rounding, replayed twice."""
    import gla

    n = 200
    A = gla.colmajor(_cov(n, np.random.default_rng(5)))
    W, tau = A.clone(), torch.zeros(n - 1, dtype=torch.float64, device="cuda")
    F0 = gla.symtri_(gla.Hermitian(A.clone(), "L"))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        gla.symtri_(gla.Hermitian(W, "L"), tau)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gla.symtri_(gla.Hermitian(W, "L"), tau)
    for _ in range(2):
        W.copy_(A)
        graph.replay()
        torch.cuda.synchronize()
        assert rel(gla.to_numpy(W), gla.to_numpy(F0.factors)) <= 1e-11
        assert rel(tau.cpu().numpy(), F0.tau.cpu().numpy()) <= 1e-10


def test_streams_follow_one_another():
    """Four threads, each with a handle and a stream of its own, reduce at once;
    every result is the one a lone call gives, bit for bit."""
    import gla

    n, reps = 1200, 3
    lib = gla.lib()
    As = [gla.colmajor(_cov(n, np.random.default_rng(i))) for i in range(4)]
    refs = []
    for A in As:
        W = A.clone()
        refs.append(gla.symtri_(gla.Hermitian(W, "L")).factors)
    torch.cuda.synchronize()
    bad = []

    def work(i):
        h = C.c_void_p()
        assert lib.gla_handle_create(C.byref(h)) == 0
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(reps):
                W = As[i].clone()
                tau = torch.zeros(n - 1, dtype=torch.float64, device="cuda")
                rc = lib.gla_symtri_d(h, b"L", n, C.c_void_p(W.data_ptr()), n,
                                      C.c_void_p(tau.data_ptr()), C.c_void_p(s.cuda_stream))
                s.synchronize()
                if rc != 0 or not torch.equal(W, refs[i]):
                    bad.append((i, rc))
        assert lib.gla_handle_destroy(h) == 0

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for th in ts:
        th.start()
    for th in ts:
        th.join()
    assert not bad


def test_wait_gives_up():
    import gla

    A = gla.colmajor(_cov(1500, np.random.default_rng(1)))
    with gla.tuning(spin_limit=1):
        F = gla.symtri_(gla.Hermitian(A.clone(), "L"))
        torch.cuda.synchronize()
        assert not torch.isfinite(F.tau).all()
    F = gla.symtri_(gla.Hermitian(A.clone(), "L"))
    assert torch.isfinite(F.tau).all()
