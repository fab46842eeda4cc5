"""symtri!, bidiagonalize! and complex QR under stream capture on a handle whose
workspace holds what the launch-per-column forms need, which are what a capture
records, but not the exchange of the one-launch forms: nothing is allocated,
which would end the capture.  Replays keep the matrix's Frobenius norm, which orthogonal transformations do,
to 10·n·eps."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _p(t):
    return C.c_void_p(t.data_ptr())


def _symtri(lib, h, W, x, s):
    n = W.shape[0]
    return lib.gla_symtri_d(h, b"L", n, _p(W), n, _p(x), s)


def _bidiag(lib, h, W, x, s):
    n, m = W.shape                                    # W: the columns, contiguous
    return lib.gla_bidiag_d(h, m, n, _p(W), m, _p(x), C.c_void_p(x.data_ptr() + 8 * n), s)


def _zqr(lib, h, W, x, s):
    n, m = W.shape
    return lib.gla_qr_blocked_z(h, m, n, _p(W), m, 32, _p(x), s)


@pytest.mark.parametrize("call,shape", [(_symtri, (2048, 2048)), (_bidiag, (2048, 2048)),
                                        (_zqr, (2048, 4096))])
def test_captured_call_needs_no_more(call, shape):
    import gla

    lib = gla.lib()
    dt = torch.complex128 if call is _zqr else torch.float64
    A = torch.randn(*shape, dtype=dt, device="cuda")
    if call is _symtri:
        A = A + A.t()
    W, x = A.clone(), torch.zeros(2 * shape[0], dtype=dt, device="cuda")
    s = torch.cuda.Stream()
    h = C.c_void_p()
    assert lib.gla_handle_create(C.byref(h)) == 0
    try:
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            cs = C.c_void_p(s.cuda_stream)
            small = A[:40, :40].clone()
            assert call(lib, h, small, torch.zeros(80, dtype=dt, device="cuda"), cs) == 0
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            rc = call(lib, h, W, x, cs)
        assert rc == 0
        for _ in range(2):
            W.copy_(A)
            g.replay()
            torch.cuda.synchronize()
            if call is _zqr:                          # W holds the columns as rows
                got = torch.tril(W[:, :shape[0]]).norm()
            else:
                d, e = W.diagonal(), W.diagonal(1 if call is _symtri else -1)
                got = (d.square().sum() + (2 if call is _symtri else 1) * e.square().sum()).sqrt()
            assert abs(got - A.norm()) <= 10 * max(shape) * 2.2e-16 * A.norm()
    finally:
        torch.cuda.synchronize()
        lib.gla_handle_destroy(h)
