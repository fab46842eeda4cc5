"""An input element with the bits of the signalling NaN that the one-launch
kernels fill their exchanges with (bidiagonalize!, src/svd.jl:321-375; symtri!,
src/eigenSelfAdjoint.jl:456-509; qrBlocked! of complex matrices,
src/qr.jl:113-146): it is taken as any NaN, and no wait runs to its limit, which
is 2^22 polls here, of at least a tenth of a microsecond each."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MARK = {torch.float64: (torch.int64, 0xFFF4C0DEC0DEC0DE - 2**64),
        torch.float32: (torch.int32, 0xFFA5C0DE - 2**32)}


def _bidiag(gla, W):
    F = gla.bidiagonalize_(W)
    return F.factors, F.taul, F.taur


def _symtri(gla, W):
    F = gla.symtri_(gla.Hermitian(W, "L"))
    return F.factors, F.tau


def _zqr(gla, W):
    F = gla.qrBlocked_(W, 32)
    return torch.view_as_real(F.factors), torch.view_as_real(F.tau)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("at", [(0, 0), (1, 0), (200, 150)])
@pytest.mark.parametrize("op", [_bidiag, _symtri, _zqr])
def test_mark_bits_in_the_input(op, at, dtype):
    import gla

    it, bits = MARK[dtype]
    m, n = (300, 300) if op is _symtri else (300, 200)
    rng = np.random.default_rng(1)
    A = torch.from_numpy(rng.standard_normal((n, m))).to(dtype).cuda()
    if op is _symtri:
        A = A + A.t()
    if op is _zqr:
        A = torch.complex(A, A.clone()).contiguous()

    def matrix(special):
        W = A.clone()
        flat = torch.view_as_real(W)[at[1], at[0], 1:] if op is _zqr else W[at[1], at[0]:at[0] + 1]
        if special:
            flat.view(it).fill_(bits)
        else:
            flat.fill_(float("nan"))
        return W.t()

    want = [torch.isnan(x) for x in op(gla, matrix(False))]
    W = matrix(True)
    with gla.tuning(spin_limit=1 << 22):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        got = op(gla, W)
        torch.cuda.synchronize()
        assert time.perf_counter() - t0 < 0.2
    for g, w in zip(got, want):
        assert torch.equal(torch.isnan(g), w)
