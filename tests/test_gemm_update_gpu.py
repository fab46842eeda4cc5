"""C − A B with enough 128×128 tiles to fill the device, K around the length
below which the product runs in 64×64 tiles, ragged edges, C a view: against a
product in 64 bits.  Bar: |C − ref| ≤ (K + 2) eps (|C0| + |A| |B|) elementwise,
a sum of K + 1 terms in any order."""
import numpy as np
import pytest

from conftest import eps_of

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("tb", ["N", "T"])
@pytest.mark.parametrize("m,n,k", [(2561, 2499, 1), (2561, 2499, 255), (2560, 2496, 256),
                                   (2497, 2559, 257), (2561, 2499, 17)])
def test_update(m, n, k, tb, dtype):
    import gla

    tdt = torch.float64 if dtype == np.float64 else torch.float32
    g = torch.Generator(device="cuda").manual_seed(k)

    def rnd(r, c):
        big = torch.randn(c, r + 3, dtype=tdt, device="cuda", generator=g).t()
        return big, big[1:1 + r, :]

    _, A = rnd(m, k)
    _, B = rnd(k, n) if tb == "N" else rnd(n, k)
    big, C = rnd(m, n)
    big0 = big.clone()
    gla.gemm_("N", tb, -1.0, A, B, 1.0, C)
    a, b = A.double().contiguous(), (B if tb == "N" else B.t()).double().contiguous()
    c0 = big0[1:1 + m, :].double()
    tol = (k + 2) * eps_of(dtype) * (c0.abs() + a.abs() @ b.abs())
    assert bool(((C.double() - (c0 - a @ b)).abs() <= tol).all())
    assert torch.equal(big[0], big0[0]) and torch.equal(big[1 + m:], big0[1 + m:])
