"""bidiagonalize! with the matrix held in registers (up to 256 blocks of 128×128):
shapes around a block's edge and around the limit, tall and wide, against the
oracle and the singular values; the same call under stream capture, which takes
the launch-per-column kernels; and a wait that gives up."""
import numpy as np
import pytest

import oracle as O
from conftest import eps_of, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m,n", [(3, 2), (127, 3), (128, 9), (129, 10), (257, 128), (256, 129),
                                 (385, 127), (9, 128), (130, 140)])
def test_shapes_vs_oracle(m, n):
    """Within 10·max(m,n)·eps of the reference in __float128, or no further
    from it than twice the FP64 oracle; a view with a leading dimension of its
    own, whose other rows stay."""
    import gla

    A = np.random.default_rng(1000 * m + n).standard_normal((m, n))
    big = gla.empty_colmajor(m + 5, n)
    big.fill_(7.0)
    X = big[3:3 + m, :]
    X.copy_(torch.from_numpy(A))
    F = gla.bidiagonalize_(X)
    got = gla.to_numpy(F.factors), F.taul.cpu().numpy(), F.taur.cpu().numpy()
    tol = 10 * max(m, n) * eps_of(np.float64)
    for g, r, t in zip(got, O.bidiag(A), O.bidiag_quad(A)):
        assert rel(g, t) <= max(tol, 2 * rel(r, t))
    rest = gla.to_numpy(big)
    assert (rest[:3] == 7).all() and (rest[3 + m:] == 7).all()


@pytest.mark.parametrize("m,n", [(2049, 2048), (2048, 2048), (8192, 200), (8300, 200),
                                 (2200, 1900), (1900, 2200)])
def test_at_the_limit(m, n):
    """Bidiagonal with the singular values of A: within 10·max(m,n)·eps·σ₁."""
    import gla

    A = np.random.default_rng(m + n).standard_normal((m, n))
    F = gla.bidiagonalize_(gla.colmajor(A))
    d, e = (x.cpu().numpy() for x in F.bidiagonal)
    B = np.diag(d) + np.diag(e, 1 if m >= n else -1)
    sa = np.linalg.svd(A, compute_uv=False)
    sb = np.linalg.svd(B, compute_uv=False)
    assert np.max(np.abs(sa - sb)) <= 10 * max(m, n) * eps_of(np.float64) * sa[0]


def test_zero_columns_and_rows():
    """Reflectors of nothing: τ = 0, as the oracle has it."""
    import gla

    A = np.random.default_rng(3).standard_normal((150, 140))
    A[:, 0] = 0
    A[5, :] = 0
    A[:, 130:] = 0
    F = gla.bidiagonalize_(gla.colmajor(A))
    ref, tl, tr = O.bidiag(A)
    assert F.taul.cpu().numpy()[0] == 0 and tl[0] == 0
    assert np.isfinite(gla.to_numpy(F.factors)).all()
    Z = np.zeros((140, 130))
    F = gla.bidiagonalize_(gla.colmajor(Z))
    assert not gla.to_numpy(F.factors).any()
    assert not F.taul.cpu().numpy().any() and not F.taur.cpu().numpy().any()


def test_captured_call_takes_the_launches():
    """Under capture the launch-per-column kernels run: the same reduction to
    rounding, replayed twice."""
    import gla

    m, n = 300, 150
    A = gla.colmajor(np.random.default_rng(5).standard_normal((m, n)))
    W = A.clone()
    F0 = gla.bidiagonalize_(A.clone())
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        gla.bidiagonalize_(W)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        F = gla.bidiagonalize_(W)
    for _ in range(2):
        W.copy_(A)
        graph.replay()
        torch.cuda.synchronize()
        assert rel(gla.to_numpy(W), gla.to_numpy(F0.factors)) <= 1e-11
        assert rel(F.taul.cpu().numpy(), F0.taul.cpu().numpy()) <= 1e-10


def test_wait_gives_up():
    import gla

    A = gla.colmajor(np.random.default_rng(1).standard_normal((1500, 900)))
    with gla.tuning(spin_limit=1):
        F = gla.bidiagonalize_(A.clone())
        torch.cuda.synchronize()
        assert not torch.isfinite(F.taul).all()
    F = gla.bidiagonalize_(A.clone())
    assert torch.isfinite(F.taul).all()
