"""The one-launch panel of the complex QR (src/qr.jl:86-146 with complex
reflectors) at its edges, against LAPACK zgeqrf at 10·max(m, n)·eps: panel
widths around 64, rows around the 128 of a workgroup, the look-ahead driver
with ragged last panels, matrices too tall for the panel, zero columns; T of
the panels through the factors' own block reflector; and a wait that gives up,
which makes the result NaN."""
import numpy as np
import pytest
import scipy.linalg as sl

from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _mat(rng, m, n, dtype):
    return (rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))).astype(dtype)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("m,n", [(2, 1), (65, 63), (129, 64), (128, 65), (127, 66), (257, 129),
                                 (300, 193), (64, 200), (1025, 320), (16300, 70)])
def test_panel_edges(rng, dtype, m, n):
    import gla

    A = _mat(rng, m, n, dtype)
    F = gla.qrBlocked_(gla.colmajor(A), 32)
    (ref, tau), _ = sl.qr(A.astype(np.complex128), mode="raw")
    k = min(m, n)
    tol = 10 * max(m, n) * eps_of(dtype)
    kk = k - 1 if m <= n else k      # LAPACK leaves a last column of length one alone
    got = gla.to_numpy(F.factors)
    assert rel(got[:, :kk], ref[:, :kk]) <= tol
    assert rel(F.tau.cpu().numpy()[:kk], tau[:kk]) <= tol
    assert rel(np.abs(np.triu(got[:k])), np.abs(np.triu(ref[:k]))) <= tol


def test_zero_columns(rng):
    """A zero column has τ = 0 and stays; the others are unaffected by it."""
    import gla

    A = _mat(rng, 300, 80, np.complex128)
    A[:, 5] = 0
    F = gla.qrBlocked_(gla.colmajor(A), 32)
    tau = F.tau.cpu().numpy()
    got = gla.to_numpy(F.factors)
    assert tau[5] == 0 and np.all(got[6:, 5] == 0)
    R = np.triu(got[:80])
    assert rel(R.conj().T @ R, A.conj().T @ A) <= 10 * 300 * eps_of(np.float64)


def test_wait_gives_up(rng):
    import gla

    A = gla.colmajor(_mat(rng, 4096, 64, np.complex128))
    with gla.tuning(spin_limit=1):
        F = gla.qrBlocked_(A.clone().t().contiguous().t(), 32)
        torch.cuda.synchronize()
        assert not torch.isfinite(torch.view_as_real(F.tau)).all()
    F = gla.qrBlocked_(A, 32)
    assert torch.isfinite(torch.view_as_real(F.factors)).all()
