"""The refined solve at the edges of the residual's 64-row blocks and rectangles
and on both sides of the order at which their size changes, and the triangle swap
of the upper convention at the edges of its tiles.  Bars: the backward error the
call was asked for (formed here in another order, hence twice it); the swap moves
values, so a factor of the mirrored matrix has to come out mirrored."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _spd(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    B = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    A = (B + B.t()) / (4 * n ** 0.5)
    A.diagonal().add_(3.0)
    return A


@pytest.mark.parametrize("n,nrhs", [(1, 1), (63, 2), (64, 16), (65, 17), (127, 1), (129, 3),
                                    (193, 1), (321, 33), (8193, 2)])
def test_refined_solve(n, nrhs):
    import gla

    A = _spd(n, n)
    g = torch.Generator(device="cuda").manual_seed(1)
    B = gla.colmajor(torch.randn(n, nrhs, dtype=torch.float64, device="cuda", generator=g))
    low = gla.colmajor(torch.tril(A) + torch.triu(torch.full_like(A, float("nan")), 1))
    X, _ = gla.chol_solve_mixed(low, B, precision="auto", tol=1e-13)
    r = torch.linalg.vector_norm(A @ X.contiguous() - B, dim=0)
    den = torch.linalg.matrix_norm(A) * torch.linalg.vector_norm(X, dim=0) + torch.linalg.vector_norm(B, dim=0)
    assert float((r / den).max()) <= 2e-13


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 200])
def test_upper_factor_mirrors_lower(n, dtype):
    import gla

    A = _spd(n, n).to(dtype)
    low = gla.colmajor(torch.tril(A) + torch.triu(torch.full_like(A, 5.0), 1))
    up = gla.colmajor(torch.triu(A) + torch.tril(torch.full_like(A, 5.0), -1))
    L = gla.cholRecursive_(low, "L").data
    U = gla.cholRecursive_(up, "U").data
    assert torch.equal(U.t(), L)
