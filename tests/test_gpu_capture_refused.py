"""The frame loops fork to the plan's own streams and are not for a caller's graph: on a capturing
stream they return an error before they enqueue anything, the capture goes on, and the plan works
after it."""
import pytest
import torch

from test_gpu_one_group import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frames", [1, 40])   # one frame group and several
def test_frame_loops_refuse_capture(gpu, rad, frames):
    from mdsf import _lib
    plan, coords, args = _system(rad, frames)
    types, scale, box, arith, wrap = args
    plan.reset()
    plan.accumulate_frames(coords.clone(), types, scale, box, arith, wrap)
    want = plan.sf()
    dsf = torch.ones(plan.half_shape, dtype=torch.float64, device="cuda")
    grad = torch.full(tuple(coords.shape), 7.0, dtype=torch.float64, device="cuda")
    work, counter, before = coords.clone(), torch.zeros(4, device="cuda"), coords.clone()
    plan.reset()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    codes = []
    with torch.cuda.graph(graph):
        counter.add_(1.0)
        common = (plan._handle, plan._ptr(work), _lib.F32, frames, plan._ptr(types), plan._ptr(scale),
                  _lib.doubles(box), arith, int(wrap[0]), int(wrap[1]))
        codes.append(plan.lib.mdsf_accumulate_frames(*common, None, None, plan._stream()))
        message = plan.lib.mdsf_last_error()
        codes.append(plan.lib.mdsf_adjoint_frames(*common, plan._ptr(dsf), plan._ptr(grad),
                                                  plan._stream()))
    assert codes == [_lib.ERR_UNSUPPORTED] * 2
    assert b"mdsf_accumulate_frames cannot be captured" in message
    for k in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(counter, torch.full((4,), k + 1.0, device="cuda"))
    assert torch.equal(work, before) and bool((grad == 7.0).all())
    plan.accumulate_frames(work, types, scale, box, arith, wrap)
    plan.check_errors()
    assert torch.equal(plan.sf(), want)
    plan.close()
