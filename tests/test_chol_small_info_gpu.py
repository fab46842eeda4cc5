"""Orders of one diagonal block (n ≤ 128) clear info in the factor's own launch:
a failing matrix between good ones leaves nothing behind, for each algorithm,
either triangle and the first order past one block; the values against the
oracle's cholUnblocked! (src/cholesky.jl:3-15) at 10·n·eps."""
import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel, spd

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ALGOS = {
    "unblocked": lambda g, X, u: g.cholUnblocked_(X, u),
    "blocked": lambda g, X, u: g.cholBlocked_(X, u, 128),
    "blocked16": lambda g, X, u: g.cholBlocked_(X, u, 16),
    "recursive": lambda g, X, u: g.cholRecursive_(X, u),
}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("algo", sorted(ALGOS))
@pytest.mark.parametrize("n", [1, 17, 128, 129])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_info_is_cleared(rng, dtype, algo, n, uplo):
    import gla

    run = ALGOS[algo]
    A = spd(n, rng, dtype)
    ref, info = O.chol_unblocked(A)
    assert info == 0
    bad = A.copy()
    bad[n - 1, n - 1] = -1
    for _ in range(2):
        with pytest.raises(gla.DomainError, match=rf"position {n}$"):
            run(gla, gla.colmajor(bad), uplo)
        X = gla.colmajor(A)
        run(gla, X, uplo)
        out = gla.to_numpy(X)
        F = np.tril(out) if uplo == "L" else np.triu(out).T
        assert rel(F, np.tril(ref)) <= 10 * n * eps_of(dtype)
