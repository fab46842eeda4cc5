"""Complex QR (src/qr.jl:113-146) on several streams at once, where the panels'
workgroups together are more than the device holds and each panel waits for all
of its own; beside symtri!, whose launch waits the same way; and under stream
capture, where the launch-per-column form runs."""
import ctypes as C
import threading

import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _zqr(lib, h, W, tau, s):
    n, m = W.shape                                  # W: the columns, contiguous
    return lib.gla_qr_blocked_z(h, m, n, C.c_void_p(W.data_ptr()), m, 32,
                                C.c_void_p(tau.data_ptr()), s)


def _symtri(lib, h, W, tau, s):
    n = W.shape[0]
    return lib.gla_symtri_d(h, b"L", n, C.c_void_p(W.data_ptr()), n, C.c_void_p(tau.data_ptr()), s)


def _together(jobs, reps=3):
    """jobs: (call, matrix, tau).  Each alone first, then all at once, each on a
    thread with a handle and a stream of its own: the same bit for bit."""
    import gla

    lib = gla.lib()
    bad = []

    def work(call, A, tau0, ref, count):
        h = C.c_void_p()
        assert lib.gla_handle_create(C.byref(h)) == 0
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(count):
                W, tau = A.clone(), torch.zeros_like(tau0)
                rc = call(lib, h, W, tau, C.c_void_p(s.cuda_stream))
                s.synchronize()
                if ref is None:
                    assert rc == 0
                    out.append((W, tau))
                elif rc != 0 or not (torch.equal(W, ref[0]) and torch.equal(tau, ref[1])):
                    bad.append((call.__name__, tuple(A.shape), rc))
        assert lib.gla_handle_destroy(h) == 0

    torch.cuda.synchronize()
    out = []
    for call, A, tau in jobs:
        work(call, A, tau, None, 1)
    refs = list(out)
    assert len(refs) == len(jobs)
    ts = [threading.Thread(target=work, args=(*j, r, reps)) for j, r in zip(jobs, refs)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def _zjob(m, n, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    A = torch.randn(n, m, dtype=torch.complex128, device="cuda", generator=g)
    return _zqr, A, torch.zeros(min(m, n), dtype=torch.complex128, device="cuda")


def test_four_tall_panels_at_once():
    _together([_zjob(12000, 200, i) for i in range(4)])


def test_many_small_ones():
    _together([_zjob(300 + 37 * i, 90, i) for i in range(8)], reps=5)


def test_beside_symtri():
    n = 2048
    g = torch.Generator("cuda").manual_seed(9)
    S = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    S = S + S.t()
    jobs = [(_symtri, S, torch.zeros(n - 1, dtype=torch.float64, device="cuda"))] * 2
    _together(jobs + [_zjob(16000, 130, i) for i in range(2)])


def test_captured():
    import gla

    A = torch.randn(150, 400, dtype=torch.complex128, device="cuda").t()
    W = A.clone()
    tau = torch.zeros(150, dtype=torch.complex128, device="cuda")
    F0 = gla.qrBlocked_(A.clone(), 32)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        gla.qrBlocked_(W, 32)
    torch.cuda.synchronize()
    lib, h = gla.lib(), gla._handle(0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        rc = _zqr(lib, h, W.t(), tau, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    for _ in range(3):
        W.copy_(A)
        graph.replay()
        torch.cuda.synchronize()
        tol = 10 * 400 * np.finfo(np.float64).eps
        assert rel(gla.to_numpy(W), gla.to_numpy(F0.factors)) <= tol
        assert rel(tau.cpu().numpy(), F0.tau.cpu().numpy()) <= tol
        (A @ A.t()).sum().item()
