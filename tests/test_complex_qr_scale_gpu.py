"""Complex QR (src/qr.jl:86-146, reflector! of src/householder.jl) near the ends
of the exponent range, against LAPACK in ComplexF64 on the matrix scaled by a
power of two.  A column of norm ν has its squares rounded to the subnormal
spacing η, so ν² is good to δ = m η/ν²; a reflector built from it, the products
with the other columns and their update together err by 8 δ of the column at
most, and that for each of the n columns, times the matrix's condition."""
import numpy as np
import pytest
import scipy.linalg as sl

from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ETA = {np.complex64: -149, np.complex128: -1074}


def _check(A, scale, dtype, e):
    """A with its columns times `scale` factored; e: exponent of the smallest."""
    import gla

    m, n = A.shape
    X = (A * scale).astype(dtype)
    assert np.array_equal(X.astype(np.complex128) / scale, A)        # exact powers of two
    F = gla.qrBlocked_(gla.colmajor(X), 32)
    got = gla.to_numpy(F.factors).astype(np.complex128)
    (ref, tau), _ = sl.qr(A, mode="raw")
    # ‖x‖² is about 2 (m − j) 2^2e, whatever the column j
    delta = 2.0 ** (ETA[dtype] - 2 * e - 1)
    tol = (10 * m * eps_of(dtype) + 16 * n * delta) * np.linalg.cond(A)
    assert tol < 0.5
    assert np.isfinite(got).all() and torch.isfinite(torch.view_as_real(F.tau)).all()
    assert rel(np.triu(got[:n]) / scale, np.triu(ref[:n])) <= tol
    assert rel(np.tril(got, -1), np.tril(ref, -1)) <= tol
    assert rel(F.tau.cpu().numpy(), tau) <= tol


def _mat(rng, m, n):
    A = rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))
    return A.astype(np.complex64).astype(np.complex128) * np.where(np.abs(A) > 2**-8, 1, 0)


# |ξ|² below the reciprocal of the largest number and ‖x‖² subnormal; and
# ‖x‖² so large that its reciprocal is subnormal
@pytest.mark.parametrize("dtype,e", [(np.complex64, -68), (np.complex64, 59),
                                     (np.complex128, -516), (np.complex128, 507)])
@pytest.mark.parametrize("m,n", [(40, 12), (300, 70)])
def test_uniform_scale(rng, dtype, e, m, n):
    A = _mat(rng, m, n)
    if e > 0 and m > 40:
        e -= 2                                   # 600·2^2e stays below the largest number
    A = np.ldexp(np.round(np.ldexp(A.real, 10)), -10) + 1j * np.ldexp(np.round(np.ldexp(A.imag, 10)), -10)
    _check(A, np.full(n, 2.0**e), dtype, min(e, 0))


@pytest.mark.parametrize("dtype,e", [(np.complex64, -68), (np.complex128, -516)])
def test_one_small_column(rng, dtype, e):
    """The columns after a small one keep their values."""
    A = _mat(rng, 40, 12)
    A = np.ldexp(np.round(np.ldexp(A.real, 10)), -10) + 1j * np.ldexp(np.round(np.ldexp(A.imag, 10)), -10)
    scale = np.ones(12)
    scale[4] = 2.0**e
    _check(A, scale, dtype, e)
