"""The dataflow Cholesky (one workgroup per 64×64 tile) behind cholRecursive!
(src/cholesky.jl:37-55), against the oracle or LAPACK at 10·n·eps: orders
around its tile edges, leading dimensions larger than n, both triangles with
the other one holding NaN, the look-ahead driver's rectangular block columns,
the index of the first negative pivot, and the report of a wait that gives
up."""
import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel, spd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _gla():
    import gla

    return gla


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [129, 143, 191, 192, 193, 256, 257, 449, 704])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_tile_edges(rng, dtype, n, uplo):
    gla = _gla()
    A = spd(n, rng, dtype)
    ref, info = O.chol_recursive(A)
    assert info == 0
    P = A.copy()
    other = np.triu_indices(n, 1) if uplo == "L" else np.tril_indices(n, -1)
    P[other] = np.nan
    big = gla.empty_colmajor(n + 13, n, getattr(torch, np.dtype(dtype).name))   # lda = n + 13
    big.fill_(7.0)
    X = big[5:5 + n, :]
    X.copy_(torch.from_numpy(P))
    gla.cholRecursive_(X, uplo)
    out = gla.to_numpy(X)
    got = np.tril(out) if uplo == "L" else np.triu(out).T
    assert rel(got, np.tril(ref)) <= 10 * n * eps_of(dtype)
    assert np.isnan(out[other]).all()
    assert (big[:5, :] == 7.0).all() and (big[5 + n:, :] == 7.0).all()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [3073, 3200, 6300])
def test_block_columns(rng, dtype, n):
    """chol_df below n: 3072-wide block columns (the last one ragged) with the
    trailing update beside the next one."""
    gla = _gla()
    A = spd(n, rng).astype(dtype)
    X = gla.colmajor(A)
    with gla.tuning(chol_df=128):
        gla.cholRecursive_(X)
    out = gla.to_numpy(X)
    ref = np.linalg.cholesky(A.astype(np.float64))
    assert rel(np.tril(out), ref) <= 10 * n * eps_of(dtype)
    assert np.array_equal(np.triu(out, 1), np.triu(A, 1))


@pytest.mark.parametrize("k", [0, 63, 64, 79, 127, 128, 200, 320])
def test_negative_pivot_index(rng, k):
    gla = _gla()
    n = 321
    A = spd(n, rng)
    L = np.linalg.cholesky(A)
    A[k, k] -= L[k, k] ** 2 + 1.0
    with pytest.raises(gla.DomainError, match=rf"position {k + 1}$"):
        gla.cholRecursive_(gla.colmajor(A))


def test_wait_gives_up(rng):
    """One poll per wait: the launch drains and the call reports the time-out;
    the next call on the handle is sound."""
    gla = _gla()
    n = 1000
    A = spd(n, rng)
    with gla.tuning(spin_limit=1):
        with pytest.raises(gla.DeviceTimeout):
            gla.cholRecursive_(gla.colmajor(A))
    X = gla.colmajor(A)
    gla.cholRecursive_(X)
    assert rel(np.tril(gla.to_numpy(X)), np.linalg.cholesky(A)) <= 10 * n * eps_of(np.float64)
