"""FP32 gradients of xy-coupled cells keep the per-voxel gather's factors: X rounded once from FP64
however deep in the Gaussian's tail, and the products with b_x and b_y and every sum in FP64
(dens.py:299-308).  One atom and one voxel of density gradient far from it along x leave a single
product per component, compared with the FP64 plan."""
import numpy as np
import pytest
import torch

from test_adjoint_ref import monoclinic

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
# X, Y and dZ round once (1/2 each in units of U); Z = expf(-q), q <= 1.4: 1 for the exponent and 2 for
# the exponential; 2^t, |t| <= 4: 2 ln 2 for t and 2 for the exponential: 8, and as much again by half
TOL = 12 * U


@pytest.mark.parametrize("theta", [100.0, 120.0])
@pytest.mark.parametrize("side", [-1, 1])
def test_one_voxel_in_the_tail(gpu, rad, theta, side):
    from mdsf import engine
    rng = np.random.default_rng(int(theta) + side)
    box, sres = np.full(3, 30.0), 0.5
    s = engine.Setup(np.zeros((1, 1, 3)), box[None], ["O"], rad, sres, False, monoclinic(theta))
    assert list(s.N) == [60, 60, 60] and int(s.half[0][0]) == 9
    plans = [engine.Plan.from_setup(s, fft64=fp64) for fp64 in (False, True)]
    types = torch.from_numpy(s.type_index.astype(np.int32)).cuda()
    scale = torch.from_numpy(np.ascontiguousarray(s.scale)).cuda()
    for _ in range(24):
        r = rng.uniform(8.0, 22.0, 3)
        home = (r / sres).astype(int)
        cell = (home[0] + 7 * side, home[1] + 1, home[2] + 2)
        gd = torch.zeros([60, 60, 60], dtype=torch.float64, device="cuda")
        gd[cell] = 1.0
        got, want = [], []
        for plan, out in zip(plans, (got, want)):
            plan.prepare_frame(torch.from_numpy(r)[None].cuda(), types, scale, [30.0] * 3, s.arith, s.wrap)
            out.append(plan.deposit_adjoint(gd).cpu().numpy()[0])
        assert np.all(np.abs(got[0] - want[0]) <= TOL * np.abs(want[0])), (got[0], want[0])
    for plan in plans:
        plan.check_errors()
        plan.close()
