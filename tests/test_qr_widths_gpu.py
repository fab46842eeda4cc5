"""Block columns at the widths and heights where the panel changes its form (24
and 32 wide, 512 rows), alone and as the last of several, against LAPACK's QR,
which takes the same signs.  Bar: 10·m·eps·κ(A), the factors' first-order
sensitivity times an error of m·eps."""
import numpy as np
import pytest

from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n", [(40, 23), (40, 24), (31, 31), (33, 32), (64, 33), (511, 24),
                                 (512, 24), (513, 23), (700, 31), (200, 151), (640, 152),
                                 (639, 152), (300, 160), (2500, 20), (160, 159)])
def test_widths(m, n, dtype):
    import gla

    A = np.random.default_rng(m * n).standard_normal((m, n)).astype(dtype)
    F = gla.qrBlocked_(gla.colmajor(A), 64)
    ref, tau = torch.geqrf(torch.from_numpy(A.astype(np.float64)))
    ref = ref.numpy()
    if m == n:   # LAPACK leaves a square matrix's last entry, reflector! negates it (τ = 2)
        ref[-1, -1] = -ref[-1, -1]
    tol = 10 * m * eps_of(dtype) * np.linalg.cond(A.astype(np.float64))
    assert rel(gla.to_numpy(F.factors), ref) <= tol
    k = n - 1 if m == n else n
    assert rel(F.tau.cpu().numpy()[:k], tau.numpy()[:k]) <= tol
