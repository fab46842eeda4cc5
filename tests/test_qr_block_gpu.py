"""qrBlocked! without its `work` (src/qr.jl:113-146) takes block columns 128
wide whatever the block size: the same factors as with `work`, which keeps
the caller's block size, and as the oracle's, at 10·max(m, n)·eps; and least
squares with the factors against the normal equations."""
import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,bs", [(40, 13, 12), (127, 127, 12), (200, 129, 5), (129, 200, 12),
                                    (300, 257, 32), (261, 190, 64)])
def test_block_size_without_work(rng, dtype, m, n, bs):
    import gla

    A = rng.standard_normal((m, n)).astype(dtype)
    fac, tau = O.qr_blocked(A, bs)
    tol = 10 * max(m, n) * eps_of(dtype)
    work = gla.colmajor(np.zeros((bs, n), dtype=dtype))
    for w in (None, work):
        F = gla.qrBlocked_(gla.colmajor(A), bs, work=w)
        assert rel(gla.to_numpy(F.factors), fac) <= tol
        assert rel(F.tau.cpu().numpy(), tau) <= tol


@pytest.mark.parametrize("m,n,nrhs", [(5, 3, 1), (129, 128, 1), (300, 129, 17), (700, 257, 3)])
def test_least_squares(rng, m, n, nrhs):
    import gla

    A = rng.standard_normal((m, n))
    B = rng.standard_normal((m, nrhs))
    F = gla.qrBlocked_(gla.colmajor(A))
    X = gla.to_numpy(gla.qr_solve_(F, gla.colmajor(B)))
    ref = np.linalg.lstsq(A, B, rcond=None)[0]
    k = np.linalg.cond(A)
    assert rel(X, ref) <= 10 * m * k * eps_of(np.float64) * max(1.0, np.linalg.norm(B) / np.linalg.norm(A @ ref))
