"""Least squares of odd shapes, where the parts of the workspace before the
triangular solves' exchange end on one element: the exchange, read 16 bytes at a
time, starts on 16 bytes.  Against numpy at 10·m·eps·κ(A)."""
import numpy as np
import pytest

from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n", [(301, 151), (303, 129), (257, 257)])
@pytest.mark.parametrize("nrhs", [1, 3, 17])
def test_odd_shapes(rng, dtype, m, n, nrhs):
    import gla

    A = rng.standard_normal((m, n)).astype(dtype)
    if m == n:
        A += 2 * m**0.5 * np.eye(n, dtype=dtype)
    b = rng.standard_normal((m, nrhs)).astype(dtype)
    F = gla.qrBlocked_(gla.colmajor(A), 12)
    x = gla.to_numpy(gla.qr_solve_(F, gla.colmajor(b)))
    A64, b64 = A.astype(np.float64), b.astype(np.float64)
    ref = np.linalg.lstsq(A64, b64, rcond=None)[0]
    assert rel(x, ref) <= 10 * m * eps_of(dtype) * np.linalg.cond(A64)
