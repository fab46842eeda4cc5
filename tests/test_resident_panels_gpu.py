"""symtri! and bidiagonalize!, whose launches hold their matrix in the registers
of the whole chip, beside QR panels (src/qr.jl:86-146) that wait for all of
theirs, each call on a thread with a handle and a stream of its own: every
result is the one of a lone call, bit for bit."""
import ctypes as C
import threading

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _p(t):
    return C.c_void_p(t.data_ptr())


def _symtri(lib, h, W, x, s):
    n = W.shape[0]
    return lib.gla_symtri_d(h, b"L", n, _p(W), n, _p(x[0]), s)


def _bidiag(lib, h, W, x, s):
    n, m = W.shape                                  # W: the columns, contiguous
    return lib.gla_bidiag_d(h, m, n, _p(W), m, _p(x[0]), _p(x[1]), s)


def _qr(lib, h, W, x, s):
    n, m = W.shape
    return lib.gla_qr_blocked_d(h, m, n, _p(W), m, 32, _p(x[0]), None, 1, s)


# 70000×8: 137 workgroups of the column-by-column panel; 40000×64 with "qr_hr"
# 0: 157, each with a CU of its own
JOBS = {
    "symtri": (_symtri, (2048, 2048), None),
    "bidiag": (_bidiag, (2000, 2048), None),
    "narrow": (_qr, (8, 70000), None),
    "panel": (_qr, (64, 40000), 0),
}


@pytest.mark.parametrize("names", [("symtri", "narrow"), ("symtri", "bidiag", "panel"),
                                   ("bidiag", "narrow", "symtri", "symtri")])
def test_at_once(names):
    import gla

    lib = gla.lib()
    bad, refs = [], {}
    mats = {}
    for i, name in enumerate(sorted(set(names))):
        g = torch.Generator("cuda").manual_seed(i)
        A = torch.randn(*JOBS[name][1], dtype=torch.float64, device="cuda", generator=g)
        mats[name] = A + A.t() if name == "symtri" else A

    def work(name, reps):
        call, _, hr = JOBS[name]
        h = C.c_void_p()
        assert lib.gla_handle_create(C.byref(h)) == 0
        if hr is not None:
            assert lib.gla_set_tuning(h, b"qr_hr", hr) == 0
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(reps):
                W = mats[name].clone()
                x = [torch.zeros(max(W.shape), dtype=torch.float64, device="cuda") for _ in range(2)]
                rc = call(lib, h, W, x, C.c_void_p(s.cuda_stream))
                s.synchronize()
                if rc != 0:
                    bad.append((name, rc))
                elif name not in refs:
                    refs[name] = (W, *x)
                elif not all(torch.equal(a, b) for a, b in zip((W, *x), refs[name])):
                    bad.append((name, "differs"))
        assert lib.gla_handle_destroy(h) == 0

    torch.cuda.synchronize()
    for name in mats:
        work(name, 1)
    assert len(refs) == len(mats)
    ts = [threading.Thread(target=work, args=(name, 4)) for name in names]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
