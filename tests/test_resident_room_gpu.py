"""Calls whose launches wait for all of their workgroups, on more threads and
streams than the library keeps track of at once, small ones beside ones that take
the chip, each result bit for bit that of a lone call; and such a call while
another thread captures a graph."""
import ctypes as C
import threading

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _p(t):
    return C.c_void_p(t.data_ptr())


def _symtri(lib, h, W, x, s):
    n = W.shape[0]
    return lib.gla_symtri_d(h, b"L", n, _p(W), n, _p(x), s)


def _zqr(lib, h, W, x, s):
    n, m = W.shape                                    # W: the columns, contiguous
    return lib.gla_qr_blocked_z(h, m, n, _p(W), m, 32, _p(x), s)


def _matrix(call, shape, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    dt = torch.complex128 if call is _zqr else torch.float64
    A = torch.randn(*shape, dtype=dt, device="cuda", generator=g)
    return A + A.t() if call is _symtri else A


def test_more_streams_than_entries():
    """40 streams on four threads, queued without waiting in between."""
    import gla

    lib = gla.lib()
    kinds = [(_symtri, (64, 64)), (_zqr, (70, 300)), (_symtri, (300, 300)), (_zqr, (20, 3000)),
             (_symtri, (1500, 1500))]
    mats = [_matrix(c, sh, i) for i, (c, sh) in enumerate(kinds)]
    refs, bad = [], []
    for (call, _), A in zip(kinds, mats):
        W, x = A.clone(), torch.zeros(max(A.shape), dtype=A.dtype, device="cuda")
        assert call(lib, gla._handle(0), W, x, None) == 0
        torch.cuda.synchronize()
        refs.append((W, x))

    def work(t):
        hs, ss, got = [], [torch.cuda.Stream() for _ in range(10)], []
        for _ in ss:
            h = C.c_void_p()
            assert lib.gla_handle_create(C.byref(h)) == 0
            hs.append(h)
        for r in range(2):
            for q, (h, s) in enumerate(zip(hs, ss)):
                k = (q + t + r) % len(kinds)
                with torch.cuda.stream(s):
                    W, x = mats[k].clone(), torch.zeros_like(refs[k][1])
                    rc = kinds[k][0](lib, h, W, x, C.c_void_p(s.cuda_stream))
                got.append((k, rc, W, x))
        for s in ss:
            s.synchronize()
        for k, rc, W, x in got:
            if rc != 0 or not (torch.equal(W, refs[k][0]) and torch.equal(x, refs[k][1])):
                bad.append((k, rc))
        for h in hs:
            assert lib.gla_handle_destroy(h) == 0

    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_while_another_thread_captures():
    import gla

    lib = gla.lib()
    A = _matrix(_symtri, (300, 300), 1)
    x = torch.zeros(300, dtype=torch.float64, device="cuda")
    W, ref = A.clone(), A.clone()
    h = C.c_void_p()
    assert lib.gla_handle_create(C.byref(h)) == 0
    s = torch.cuda.Stream()
    cs = C.c_void_p(s.cuda_stream)
    torch.cuda.synchronize()
    for _ in range(2):                                # the workspace, and an entry to look at
        assert _symtri(lib, h, ref.copy_(A), x, cs) == 0
        torch.cuda.synchronize()
    a = torch.zeros(1000, device="cuda")
    rcs = []

    def other():
        for _ in range(3):
            rcs.append(_symtri(lib, h, W, x, cs))

    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a += 1
        t = threading.Thread(target=other)
        t.start()
        t.join()
        a += 1
    assert rcs == [0, 0, 0]
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    assert (a == 2).all()
    assert _symtri(lib, h, W.copy_(A), x, cs) == 0
    torch.cuda.synchronize()
    assert torch.equal(W, ref)
    assert lib.gla_handle_destroy(h) == 0
