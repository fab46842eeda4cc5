"""The diagonal factor's 16×16 tiles at their edges, against the oracle's
cholUnblocked! (src/cholesky.jl:3-15) at 10·n·eps: sizes around multiples of
4 (its column groups), 16 (its tiles) and 128 (its block), with the strict
upper triangle, which must not be read, holding NaN; and the index of the
first negative pivot at every place of a tile."""
import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel, spd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [4, 5, 15, 16, 17, 31, 33, 47, 97, 111, 112, 113, 126])
def test_tile_edges(rng, dtype, n):
    import gla

    A = spd(n, rng, dtype)
    ref, info = O.chol_unblocked(A)
    assert info == 0
    P = A.copy()
    P[np.triu_indices(n, 1)] = np.nan
    X = gla.colmajor(P)
    gla.cholUnblocked_(X)
    out = gla.to_numpy(X)
    assert rel(np.tril(out), np.tril(ref)) <= 10 * n * eps_of(dtype)
    assert np.isnan(out[np.triu_indices(n, 1)]).all()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("k", [0, 1, 3, 4, 7, 14, 15, 16, 18, 31, 32, 77, 111, 112, 115])
def test_negative_pivot_index(rng, dtype, k):
    import gla

    n = 116
    A = spd(n, rng)
    L = np.linalg.cholesky(A)
    A[k, k] -= L[k, k] ** 2 + 1.0
    with pytest.raises(gla.DomainError, match=rf"position {k + 1}$"):
        gla.cholUnblocked_(gla.colmajor(A.astype(dtype)))
