"""Gradient calls of one plan from several streams with no synchronisation between them: each call's
weights (dL/dS) are the plan's until its transforms have read them, so the next call waits, whether a
call is one frame group or several, with accumulating calls in between."""
import numpy as np
import pytest
import torch

from test_gpu_one_group import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("sizes", [(1, 1, 1, 1, 1), (3, 40, 1, 40, 2, 35)])
def test_each_call_keeps_its_weights(gpu, rad, sizes, fp64):
    from mdsf import _lib
    plan, coords, args = _system(rad, max(sizes), fp64)
    types, scale, box, arith, wrap = args
    g = torch.Generator("cuda").manual_seed(len(sizes))
    dsf = [10.0 ** k * torch.randn(plan.half_shape, dtype=torch.float64, device="cuda", generator=g)
           for k in range(len(sizes))]
    want = []
    for k, w in zip(sizes, dsf):
        want.append(plan.adjoint_frames(coords[:k].clone(), types, scale[:k], box, arith, wrap, w))
        torch.cuda.synchronize()
    work = [coords[:k].clone() for k in sizes]
    more = coords[:5].clone()
    got = [torch.empty(c.shape, dtype=torch.float64, device="cuda") for c in work]
    streams = [torch.cuda.Stream() for _ in sizes]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for i, (st, c, k, w, out) in enumerate(zip(streams, work, sizes, dsf, got)):
        with torch.cuda.stream(st):
            plan.adjoint_frames(c, types, scale[:k], box, arith, wrap, w, grad=out)
        if i == 2:
            with torch.cuda.stream(side):
                plan.accumulate_frames(more, types, scale[:5], box, arith, wrap)
        if i == 3:   # no frames: nothing of the plan is touched
            _lib.check(plan.lib.mdsf_adjoint_frames(
                plan._handle, plan._ptr(coords), _lib.F32, 0, plan._ptr(types), plan._ptr(scale),
                _lib.doubles(box), arith, 0, 0, plan._ptr(dsf[0]), plan._ptr(got[0]), plan._stream()))
    torch.cuda.synchronize()
    plan.check_errors()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    plan.close()
