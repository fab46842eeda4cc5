"""QR of 17 to 24 columns at the heights where the panel changes its form (1024
and 4096 (n − 17) rows, 512 for 24), against LAPACK's QR, which takes the same
signs.  Bar: 10·m·eps·κ(A), the factors' first-order sensitivity times an error
of m·eps."""
import numpy as np
import pytest

from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n", [(1100, 17), (1023, 18), (1024, 18), (4096, 18), (4097, 18),
                                 (12289, 20), (16384, 21), (24577, 23), (1030, 151)])
def test_heights(m, n, dtype):
    import gla

    A = np.random.default_rng(m * n).standard_normal((m, n)).astype(dtype)
    F = gla.qrBlocked_(gla.colmajor(A), 64)
    ref, tau = torch.geqrf(torch.from_numpy(A.astype(np.float64)))
    tol = 10 * m * eps_of(dtype) * np.linalg.cond(A.astype(np.float64))
    assert rel(gla.to_numpy(F.factors), ref.numpy()) <= tol
    assert rel(F.tau.cpu().numpy(), tau.numpy()) <= tol
