"""A wait of the complex QR panel that gives up is the panel's last: the time of
a panel whose arrivals never count is that of one wait per wave, not one per
column."""
import time

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_one_wait_gives_up_for_the_whole_panel():
    import gla

    def seconds(n):
        A = torch.randn(n, 4096, dtype=torch.complex128, device="cuda").t()
        gla.qrBlocked_(A.clone(), 64)
        torch.cuda.synchronize()
        with gla.tuning(spin_limit=1 << 14, qr_wait_test=1):
            t0 = time.perf_counter()
            F = gla.qrBlocked_(A.clone(), 64)
            torch.cuda.synchronize()
            t = time.perf_counter() - t0
        assert torch.isnan(torch.view_as_real(F.tau)).all()
        F = gla.qrBlocked_(A, 64)
        assert torch.isfinite(torch.view_as_real(F.factors)).all()
        return t

    one = seconds(1)
    assert one > 1e-3                       # 2^14 polls: it did wait
    assert seconds(64) < 4 * one
