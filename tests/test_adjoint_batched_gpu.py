"""The batched Cholesky adjoint at the edges of a 16-row tile and of the sizes
its workgroup shapes hold (32, 64, 128), against the oracle's adjoint of each
matrix's LAPACK factor; strides and leading dimensions of their own, and the
result written over L̄.  Bar: relative difference ≤ 50·n·eps, as for the single
matrix."""
import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _spd(n, rng):
    B = rng.standard_normal((n, n))
    return B.T @ B + n * np.eye(n)


def _strided(mats, tdt, ld):
    """(batch, n, n) column-major view into storage with leading dimension ld
    and a gap of ld + 3 between the matrices; 9 outside."""
    b, n = len(mats), mats[0].shape[0]
    st = torch.full((b * (n * ld + ld + 3) + 1,), 9.0, dtype=tdt, device="cuda")
    V = st.as_strided((b, n, n), (n * ld + ld + 3, 1, ld), 1)
    V.copy_(torch.from_numpy(np.stack(mats)).to(tdt))
    return st, V


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("conv", ["S", "L"])
@pytest.mark.parametrize("n", [1, 2, 15, 17, 31, 32, 33, 47, 49, 63, 64, 65, 81, 111, 127, 128])
def test_orders(n, conv, dtype):
    import gla

    tdt = torch.float64 if dtype == np.float64 else torch.float32
    rng = np.random.default_rng(n)
    As = [_spd(n, rng) for _ in range(3)]
    Ws = [rng.standard_normal((n, n)) for _ in range(3)]
    nan = np.triu(np.full((n, n), np.nan), 1)
    _, A = _strided([np.tril(a) + nan for a in As], tdt, n + 1)
    st, W = _strided([np.tril(w) + nan for w in Ws], tdt, n + 2)
    got = gla.chol_adjoint_batched(A, W, conv, out=W).cpu().numpy()
    for b in range(3):
        L = np.linalg.cholesky(As[b].astype(dtype).astype(np.float64))
        ref = O.chol_adjoint(L, np.tril(Ws[b].astype(dtype).astype(np.float64)), conv)
        assert rel(got[b], ref) <= 50 * n * eps_of(dtype)
        if conv == "S":
            assert np.array_equal(got[b], got[b].T)
        else:
            assert not np.triu(got[b], 1).any()
    W.fill_(9.0)
    assert (st == 9).all()


def test_captured_call_replays():
    import gla

    rng = np.random.default_rng(4)
    A = torch.empty((7, 100, 100), dtype=torch.float64, device="cuda").transpose(1, 2)
    W, out = torch.empty_like(A), torch.empty_like(A)
    ins = [(torch.from_numpy(np.stack([_spd(100, rng) for _ in range(7)])),
            torch.from_numpy(rng.standard_normal((7, 100, 100)))) for _ in range(3)]
    A.copy_(ins[0][0])
    W.copy_(ins[0][1])
    lib = gla.lib()
    import ctypes as C

    h = C.c_void_p()
    assert lib.gla_handle_create(C.byref(h)) == 0
    s = torch.cuda.Stream()

    def call():
        assert lib.gla_chol_adjoint_batched_d(
            h, b"S", 100, 7, C.c_void_p(A.data_ptr()), 100, 10000, C.c_void_p(W.data_ptr()), 100,
            10000, C.c_void_p(out.data_ptr()), 100, 10000, None,
            C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0

    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        call()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for a, w in ins:
        A.copy_(a)
        W.copy_(w)
        graph.replay()
        torch.cuda.synchronize()
        ref = gla.chol_adjoint_batched(A, W, "S")
        assert torch.equal(out, ref)
    torch.cuda.synchronize()
    assert lib.gla_handle_destroy(h) == 0
