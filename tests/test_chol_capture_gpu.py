"""cholRecursive! (src/cholesky.jl:37-55) under stream capture, on a handle of
its own: with the dataflow buffer in place, and where it would have to grow in
the capture, which then records the driver by launches; and replayed after an
eager call that needed a larger buffer.  Every replay, between
eager work, against the oracle at 10·n·eps."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel, spd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("warm", ["same", "blocked", "grown"])
@pytest.mark.parametrize("dtype,sfx", [(np.float64, "d"), (np.float32, "s")])
def test_capture(rng, dtype, sfx, warm):
    import gla
    from gla._lib import lib

    n = 700
    L = lib()
    A = spd(n, rng, dtype)
    ref, info = O.chol_unblocked(A)
    assert info == 0
    src = gla.colmajor(A)
    X = gla.colmajor(A)
    hp = C.c_void_p()
    assert L.gla_handle_create(C.byref(hp)) == 0
    h = hp.value
    run = getattr(L, f"gla_chol_recursive_{sfx}")

    def call(stream):
        return run(h, b"L", n, C.c_void_p(X.data_ptr()), n, 1, None, C.c_void_p(stream.cuda_stream))

    try:
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            if warm != "blocked":
                assert call(s) == 0
            else:
                rc = getattr(L, f"gla_chol_blocked_{sfx}")(
                    h, b"L", n, C.c_void_p(X.data_ptr()), n, 128, None,
                    C.c_void_p(s.cuda_stream))
                assert rc == 0
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            rc = call(s)
        assert rc == 0
        if warm == "grown":
            big = 2 * torch.eye(4000, dtype=src.dtype, device="cuda")
            assert run(h, b"L", 4000, C.c_void_p(big.data_ptr()), 4000, 1, None, _stream()) == 0
            want = 2**0.5
            err = (big.diagonal().double() - want).abs().max().item()
            assert err <= 10 * 4000 * eps_of(dtype) * want
        for _ in range(3):
            X.copy_(src)
            g.replay()
            torch.cuda.synchronize()
            assert rel(np.tril(gla.to_numpy(X)), np.tril(ref)) <= 10 * n * eps_of(dtype)
            (src @ src).sum().item()
        del g
    finally:
        torch.cuda.synchronize()
        L.gla_handle_destroy(C.c_void_p(h))
