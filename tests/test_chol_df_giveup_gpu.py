"""A wait of the dataflow Cholesky (cholRecursive!, src/cholesky.jl:37-55) that
gives up in a call that asks for no info: what it could not compute is NaN, and
what is not NaN is the factor of an undisturbed call, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from conftest import spd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [200, 1000, 2500])
@pytest.mark.parametrize("dtype,sfx", [(np.float64, "d"), (np.float32, "s")])
def test_nan_without_info(rng, dtype, sfx, n):
    import gla

    A = gla.colmajor(spd(n, rng, dtype))
    run = getattr(gla.lib(), f"gla_chol_recursive_{sfx}")
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)

    def factor():
        X = A.clone()
        assert run(gla._handle(0), b"L", n, C.c_void_p(X.data_ptr()), n, 1, None, s) == 0
        return torch.tril(X)

    ref = factor()
    assert torch.isfinite(ref).all()
    with gla.tuning(spin_limit=1):
        for _ in range(3):
            X = factor()
            lost = torch.isnan(X)
            assert lost.any()
            assert torch.equal(X[~lost], ref[~lost])
    assert torch.equal(factor(), ref)
