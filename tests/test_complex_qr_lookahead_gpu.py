"""Complex QR (src/qr.jl:113-146) on both sides of the sizes from which the next
panel is factored beside the trailing update, 4.5 million elements (ComplexF32 16
million), with ragged last block columns: RᴴR = AᴴA, and the reflectors take A to
R, to 10·m·eps."""
import pytest

from conftest import eps_of

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype,m,n", [("complex128", 2249, 2000), ("complex128", 2251, 2000),
                                       ("complex128", 1990, 2300), ("complex128", 16200, 290),
                                       ("complex64", 4010, 3985), ("complex64", 4013, 3990)])
def test_both_sides(dtype, m, n):
    import gla

    g = torch.Generator("cuda").manual_seed(m)
    A = torch.randn(n, m, dtype=getattr(torch, dtype), device="cuda", generator=g).t()
    W = A.clone()
    F = gla.qrBlocked_(W, 32)
    tol = 10 * m * eps_of("float64" if dtype == "complex128" else "float32")
    k = min(m, n)
    A, V = A.to(torch.complex128), F.factors.to(torch.complex128)
    R = torch.triu(V[:k])
    G, H = A.conj().t().contiguous() @ A.contiguous(), R.conj().t().contiguous() @ R.contiguous()
    assert (G - H).norm() <= tol * G.norm()
    # a few columns of A through all reflectors, last ones included
    cols = [0, 1, k // 2, n - 2, n - 1]
    x = A[:, cols].contiguous()
    tau = F.tau.to(torch.complex128)
    for j in range(k):
        v = V[:, j].clone()
        v[:j] = 0
        v[j] = 1
        x -= torch.outer(v, tau[j].conj() * (v.conj() @ x))
    want = torch.zeros_like(x)
    want[:k] = R[:, cols]
    assert (x - want).norm() <= tol * A[:, cols].norm()
