"""Frame groups: the frame loops hand every kernel several frames of a small grid at once.  A call
of many frames has to give bit for bit what one-frame calls give (dens.py:277-321): S(q), the
coordinates it rescales and wraps, the last frame's home cells, the occupancy and the gradients, at
frame counts around the group size (the 20^3 to 36^3 grids here take 16 frames per group)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

RAD = {"H": (1.0, 0.53), "C": (6.0, 0.7), "O": (8.0, 0.6)}
CELLS = {"orth": np.eye(3),
         "xy": np.array([[1.0, 0, 0], [-0.5, np.sqrt(0.75), 0], [0, 0, 1]]),
         "general": np.array([[1.0, 0, 0], [0.5, np.sqrt(0.75), 0], [0.5, 0.29, 0.82]])}


def _system(nframes, cell, fp64):
    from mdsf import engine
    rng = np.random.default_rng(nframes)
    box = np.array([12.0, 17.0, 14.0])
    typ = np.array(["H", "C", "O"])[rng.integers(0, 3, 150)]
    # beyond the cell on both sides too (parked atoms), and boxes that change
    coords = rng.uniform(-0.2, 1.2, size=(nframes, 150, 3)) * box
    dims = box * (1 + 0.01 * rng.normal(size=(nframes, 3)))
    s = engine.Setup(coords, dims, typ, RAD, 0.6, True, CELLS[cell])
    plan = engine.Plan.from_setup(s, fft64=fp64)
    types = torch.from_numpy(s.type_index.astype(np.int32)).cuda()
    scale = torch.from_numpy(np.ascontiguousarray(s.scale)).cuda()
    return s, plan, torch.from_numpy(coords).cuda(), types, scale, [float(x) for x in s.L]


@pytest.mark.parametrize("nframes", [2, 16, 17, 35])
@pytest.mark.parametrize("cell,fp64", [("orth", False), ("orth", True), ("xy", False),
                                       ("general", False)])
def test_frames_together_equal_frames_alone(gpu, nframes, cell, fp64):
    s, plan, coords, types, scale, box = _system(nframes, cell, fp64)
    out = []
    for step in (nframes, 1):
        c = coords.clone()
        occ = torch.zeros(plan.n, dtype=torch.int32, device="cuda")
        home = torch.zeros(plan.natoms, 3, dtype=torch.int32, device="cuda")
        plan.reset()
        for t in range(0, nframes, step):
            plan.accumulate_frames(c[t:t + step], types, scale[t:t + step], box, s.arith, s.wrap,
                                   occupancy=occ, home=home)
        plan.check_errors()
        out.append((plan.sf(), c, occ, home))
    # parked atoms add with atomics, whose order is free: FP32 sums of a few hundred terms a voxel
    torch.testing.assert_close(out[0][0], out[1][0], rtol=1e-5, atol=1e-7 * float(out[1][0].max()))
    for a, b in zip(out[0][1:], out[1][1:]):
        assert torch.equal(a, b)
    # without parked atoms
    inside = torch.remainder(coords, torch.tensor(box, device="cuda") * 0.97)
    sf = []
    for step in (nframes, 1):
        plan.reset()
        for t in range(0, nframes, step):
            plan.accumulate_frames(inside[t:t + step].clone(), types, scale[t:t + step], box, s.arith,
                                   s.wrap)
        plan.check_errors()
        sf.append(plan.sf())
    assert torch.equal(sf[0], sf[1])
    plan.close()


@pytest.mark.parametrize("cell,fp64", [("orth", False), ("orth", True), ("xy", False)])
def test_gradients_together_equal_gradients_alone(gpu, cell, fp64):
    nframes = 19
    s, plan, coords, types, scale, box = _system(nframes, cell, fp64)
    inside = torch.remainder(coords, torch.tensor(box, device="cuda") * 0.97)
    g = torch.randn(plan.half_shape, dtype=torch.float64, device="cuda",
                    generator=torch.Generator("cuda").manual_seed(3))
    grads = []
    for step in (nframes, 1):
        grads.append(torch.cat([plan.adjoint_frames(inside[t:t + step].clone(), types,
                                                    scale[t:t + step], box, s.arith, s.wrap, g)
                                for t in range(0, nframes, step)]))
    plan.check_errors()
    assert float(grads[1].abs().max()) > 0
    assert torch.equal(grads[0], grads[1])
    plan.close()
