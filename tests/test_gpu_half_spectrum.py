"""The reorder between the accumulators' [kz][ky][kx] half spectrum and the reference's
[kx][ky][kz] at the edges of its tiles (32 kx by 64 kz): S(q), the spectrum and the adjoint
weights of FP64 plans against torch's FP64 transform (dens.py:313-318)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# an FP64 transform of n <= 2^16 points: a few eps log2(n) of the largest bin
TOL = 64 * 2.0 ** -53


@pytest.mark.parametrize("n", [(2, 2, 2), (32, 4, 126), (34, 6, 128), (66, 2, 2), (30, 10, 130),
                               (64, 2, 254)])
def test_half_spectrum_layouts(gpu, n):
    from mdsf import engine
    plan = engine.Plan(n, 0, [1.0] * 3, np.eye(3), [], [], [], [], fft64=True)
    g = torch.Generator().manual_seed(sum(n))
    d = torch.rand(n, dtype=torch.float64, generator=g).requires_grad_(True)
    want = torch.fft.rfftn(d)
    got = plan.rfft3(d.detach()).cpu()
    top = float(want.detach().abs().max())
    assert float((got - want).abs().max()) <= TOL * top
    plan.reset()
    plan.accumulate_density(d.detach())
    s = want.abs().square()
    assert float((plan.sf().cpu() - s.detach()).abs().max()) <= 2 * TOL * float(s.detach().max())
    w = torch.randn(s.shape, dtype=torch.float64, generator=g)
    (s * w).sum().backward()
    grad = plan.density_adjoint(d.detach(), w).cpu()
    # the inverse adds n bins, each to a few eps log2(n) of the largest weighted bin
    bound = 2 * TOL * 2 * float((w * want.detach().abs()).abs().sum())
    assert float((grad - d.grad).abs().max()) <= bound
    plan.close()
