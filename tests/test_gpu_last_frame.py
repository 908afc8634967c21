"""After a frame loop the single-frame entry points find its last frame in the plan's slot, whatever
the frame groups: the density deposited again, the gradient of a given density gradient, the slot
selected again (dens.py:283-311)."""
import pytest
import torch

from test_gpu_frame_groups import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nframes", [1, 5, 16, 20])
@pytest.mark.parametrize("cell,fp64", [("orth", False), ("orth", True), ("xy", False), ("xy", True),
                                       ("general", False), ("general", True)])
def test_last_frame_stays(gpu, nframes, cell, fp64):
    from mdsf import engine
    s, plan, coords, types, scale, box = _system(nframes, cell, fp64)
    inside = torch.remainder(coords, torch.tensor(box, device="cuda") * 0.97)
    args = (types, scale, box, s.arith, s.wrap)
    last = (types, scale[-1], box, s.arith, s.wrap)
    other = engine.Plan.from_setup(s, fft64=fp64, max_frames=1)
    want = other.deposit_fold(inside[-1].clone(), *last)
    gd = torch.randn(plan.n, dtype=plan.real_dtype, device="cuda",
                     generator=torch.Generator("cuda").manual_seed(1))
    out = torch.empty_like(want)
    plan.accumulate_frames(inside.clone(), *args)
    plan.deposit(out)
    assert torch.equal(out, want)
    if cell != "general":
        grad = other.deposit_adjoint(gd)
        assert torch.equal(plan.deposit_adjoint(gd), grad)      # (its buffers are made here)
        dsf = torch.ones(plan.half_shape, dtype=torch.float64, device="cuda")
        plan.adjoint_frames(inside.clone(), *args, dsf)
        assert torch.equal(plan.deposit_adjoint(gd), grad)
        plan.deposit(out)
        assert torch.equal(out, want)
    slot = ((nframes + 15) // 16 - 1) % 3                       # groups of 16 here
    plan.set_frame_buffer((slot + 1) % 3)
    plan.set_frame_buffer(slot)
    plan.deposit(out)
    assert torch.equal(out, want)
    # a frame prepared there afterwards, and another loop
    plan.prepare_frame(inside[0].clone(), types, scale[0], box, s.arith, s.wrap)
    plan.deposit(out)
    assert torch.equal(out, other.deposit_fold(inside[0].clone(), types, scale[0], box, s.arith, s.wrap))
    plan.reset()
    plan.accumulate_frames(inside.clone(), *args)
    other.reset()
    other.accumulate_frames(inside.clone(), *args)
    assert torch.equal(plan.sf(), other.sf())
    plan.check_errors()
    plan.close()
    other.close()
