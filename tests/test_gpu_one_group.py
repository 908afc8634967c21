"""Frame loops of one group run on the caller's stream alone; the plan's calls stay in order whatever
streams they come from."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _system(rad, frames, fp64=False, n=300):
    from mdsf import engine
    rng = np.random.default_rng(frames)
    box = np.array([14.0, 13.0, 12.0])
    coords = (rng.random((frames, n, 3)) * box).astype(np.float32)
    s = engine.Setup(coords, np.tile(box, (frames, 1)), ["C", "O", "H"] * (n // 3), rad, 0.5, False,
                     np.eye(3))
    plan = engine.Plan.from_setup(s, fft64=fp64)
    types = torch.from_numpy(s.type_index.astype(np.int32).reshape(-1)).to(plan.device)
    scale = torch.from_numpy(np.ascontiguousarray(s.scale, dtype=np.float64)).to(plan.device)
    args = (types, scale, [float(v) for v in s.L], s.arith, s.wrap)
    return plan, torch.from_numpy(coords).to(plan.device), args


@pytest.mark.parametrize("sizes", [(1, 1, 1, 1), (3, 40, 2, 40, 1)])
def test_calls_from_several_streams(gpu, rad, sizes):
    """Calls of one group and of several, each from another stream with no synchronisation."""
    plan, coords, args = _system(rad, max(sizes))
    types, scale, box, arith, wrap = args
    want = torch.zeros(plan.half_shape, dtype=torch.float64, device=plan.device)
    for k in sizes:
        plan.reset()
        plan.accumulate_frames(coords[:k].clone(), types, scale[:k], box, arith, wrap)
        torch.cuda.synchronize()
        want += plan.sf()
    torch.cuda.synchronize()
    plan.reset()
    work = [coords[:k].clone() for k in sizes]
    streams = [torch.cuda.Stream() for _ in sizes]
    torch.cuda.synchronize()
    for st, c, k in zip(streams, work, sizes):
        with torch.cuda.stream(st):
            plan.accumulate_frames(c, types, scale[:k], box, arith, wrap)
    torch.cuda.synchronize()
    plan.check_errors()
    # sums of positive values in another grouping
    torch.testing.assert_close(plan.sf(), want, rtol=1e-13, atol=0)
