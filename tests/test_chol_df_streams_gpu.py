"""cholRecursive! (src/cholesky.jl:37-55) by the dataflow launch on several
streams at once, with more workgroups than the device holds between them, and
beside symtri!, which holds every CU: each call on a thread with a handle and a
stream of its own, every factor bit for bit that of a lone call."""
import ctypes as C
import threading

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _p(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("sizes,symtri", [((3000, 3000, 2500, 2500), 0), ((8192, 8192), 0),
                                          ((3000, 2500), 2), ((9000, 3000, 1000, 700), 1)])
def test_at_once(sizes, symtri):
    import gla

    lib = gla.lib()
    bad = []

    def call(lib, h, A, s):
        n = A.shape[0]
        W = A.clone()
        if A.dtype == torch.float32:                 # the matrix of a symtri!
            W = W.double()
            tau = torch.zeros(n, dtype=torch.float64, device="cuda")
            return W, lib.gla_symtri_d(h, b"L", n, _p(W), n, _p(tau), s)
        return W, lib.gla_chol_recursive_d(h, b"L", n, _p(W), n, 1, None, s)

    def work(A, ref, out, reps):
        h = C.c_void_p()
        assert lib.gla_handle_create(C.byref(h)) == 0
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(reps):
                W, rc = call(lib, h, A, C.c_void_p(s.cuda_stream))
                s.synchronize()
                if out is not None:
                    out.append(W)
                if rc != 0 or (ref is not None and not torch.equal(W, ref)):
                    bad.append((tuple(A.shape), rc))
        assert lib.gla_handle_destroy(h) == 0

    mats = []
    for i, n in enumerate((*sizes, *[2048] * symtri)):
        g = torch.Generator("cuda").manual_seed(i)
        B = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
        B = B + B.t()
        mats.append(B.float() if i >= len(sizes) else B + 4 * n**0.5 * torch.eye(n, device="cuda"))
    torch.cuda.synchronize()
    refs = []
    for A in mats:
        work(A, None, refs, 1)
    assert not bad
    assert all(torch.isfinite(r).all() for r in refs)
    ts = [threading.Thread(target=work, args=(A, r, None, 4)) for A, r in zip(mats, refs)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
