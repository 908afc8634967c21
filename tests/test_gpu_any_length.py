"""The any-length FFT passes where they can go wrong: every radix as first, middle and last stage,
primes above 13 alone and with other factors, one to four stages, partial tiles of pencils, the
longest, and the lengths next to them that keep the LDS-staged pass -- forward, inverse (the
adjoint's) and accumulating, against torch's FP64 transform (dens.py:313-318)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53
# x, y and z lengths (the z pass transforms half of the last): each tuple mixes short and long so
# that every length passes through the x (along rows), y (across) and z kernels once
LENGTHS = [6, 10, 12, 14, 18, 20, 22, 26, 28, 30, 34, 38, 46, 58, 74, 82, 90, 104, 106, 110, 130, 154,
           180, 182, 208, 210, 220, 226, 242, 250, 254, 286, 338, 390, 420, 500, 586, 720, 822, 1014,
           1018, 1022]
FALLBACK = [578, 722, 900, 1026, 1100]     # 2 17^2, 2 19^2, 10 9 10 (a middle radix above 8), > 1024


def _check(n, fp64=True):
    from mdsf import engine
    plan = engine.Plan(n, 0, [1.0] * 3, np.eye(3), [], [], [], [], fft64=fp64)
    g = torch.Generator().manual_seed(sum(n))
    d = torch.rand(n, dtype=torch.float64, generator=g) - 0.5
    if not fp64:
        d = d.float().double()
    want = torch.fft.rfftn(d)   # on the host
    top = float(want.abs().max())
    # direct DFTs of primes up to 509 add 254 products: (n_x + n_y + n_z) eps of the largest bin
    # bounds every stage; FP32 storage adds half an ulp (2^-24) of each pass's values, spread by the
    # next pass over sqrt(n) bins
    tol = sum(n) * EPS if fp64 else 3 * 2.0 ** -24
    got = plan.rfft3(d).cpu()
    assert float((got - want).abs().max()) <= tol * top * (1 if fp64 else 4)
    s = want.abs().square()
    plan.reset()
    plan.accumulate_density(d)
    plan.accumulate_density(d)
    assert float((plan.sf().cpu() - 2 * s).abs().max()) <= 16 * tol * float(s.max())
    if fp64:
        w = torch.randn(s.shape, dtype=torch.float64, generator=g)
        x = d.clone().requires_grad_(True)
        (torch.fft.rfftn(x).abs().square() * w).sum().backward()
        grad = plan.density_adjoint(d, w).cpu()
        bound = 4 * sum(n) * EPS * float((w * want).abs().square().sum().sqrt()) * 4
        assert float((grad - x.grad).abs().max()) <= bound
    plan.close()


@pytest.mark.parametrize("n", LENGTHS + FALLBACK)
def test_each_length_on_each_axis(gpu, n):
    _check((n, 6, 4))
    _check((6, n, 10))
    if n <= 1022:
        _check((4, 18, 2 * n))


@pytest.mark.parametrize("n", [(104, 90, 80), (106, 92, 82), (30, 34, 38), (18, 250, 26)])
def test_fp32_plans(gpu, n):
    _check(n, fp64=False)


@pytest.mark.parametrize("nx,ny", [(16, 16), (16, 512), (512, 16), (64, 1024), (1024, 64), (32, 256),
                                   (256, 128), (512, 512), (1024, 1024), (64, 90), (90, 64)])
def test_residual_blocks(gpu, nx, ny):
    """FP32 plans of power-of-two lengths pass the y pass's residuals in blocks of x: every width
    next to lengths that keep rows."""
    _check((nx, ny, 4), fp64=False)
