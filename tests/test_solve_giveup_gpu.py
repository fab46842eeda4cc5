"""Least squares (src/qr.jl:64-83 and a triangular solve) whose device-side wait
gives up: the call, which synchronises, reports it; the next one is sound."""
import numpy as np
import pytest

from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_least_squares_reports(rng, dtype):
    import gla

    m, n = 2000, 1500
    A = rng.standard_normal((m, n)).astype(dtype)
    b = rng.standard_normal((m, 1)).astype(dtype)
    F = gla.qrBlocked_(gla.colmajor(A), 32)
    with gla.tuning(spin_limit=1):
        with pytest.raises(gla.DeviceTimeout, match="gave up"):
            gla.qr_solve_(F, gla.colmajor(b))
    x = gla.to_numpy(gla.qr_solve_(F, gla.colmajor(b)))
    A64, b64 = A.astype(np.float64), b.astype(np.float64)
    ref = np.linalg.lstsq(A64, b64, rcond=None)[0]
    assert rel(x, ref) <= 10 * m * eps_of(dtype) * np.linalg.cond(A64)
