"""cholRecursive! (src/cholesky.jl:37-55) of orders above a lowered "chol_df"
and up to the width of a dataflow block column: the drivers without the tile
buffer run, which is neither taken, grown nor given back.  Against LAPACK at
10·n·eps, on a handle of its own."""
import ctypes as C

import numpy as np
import pytest

from conftest import eps_of, rel, spd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("warm", [0, 1000])
@pytest.mark.parametrize("n", [129, 200, 1000, 2000, 3072])
def test_between_chol_df_and_a_block_column(rng, n, warm):
    import gla

    L = gla.lib()
    A = spd(n, rng)
    h = C.c_void_p()
    assert L.gla_handle_create(C.byref(h)) == 0
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)

    def chol(name, X, *extra):
        info = C.c_int64(-1)
        k = X.shape[0]
        rc = getattr(L, name)(h, b"L", k, C.c_void_p(X.data_ptr()), k, *extra, C.byref(info), s)
        assert rc == 0 and info.value == 0

    try:
        X = gla.colmajor(A)
        chol("gla_chol_blocked_d", X, 128)                     # the workspace
        if warm:
            chol("gla_chol_recursive_d", gla.colmajor(spd(warm, rng)), 1)
        X = gla.colmajor(A)
        assert L.gla_set_tuning(h, b"chol_df", 128) == 0
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
        chol("gla_chol_recursive_d", X, 1)
        assert torch.cuda.mem_get_info()[0] == free0
        assert rel(np.tril(gla.to_numpy(X)), np.linalg.cholesky(A)) <= 10 * n * eps_of(np.float64)
    finally:
        torch.cuda.synchronize()
        L.gla_handle_destroy(h)
