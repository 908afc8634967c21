"""The FP32 adjoint from the tile lists at the edges of its batches (64 regular atoms of a tile, 16
corner atoms) against the FP64 plan's gather of the same density gradient (pinned to autograd in
test_gpu_adjoint.py), orthogonal and xy-coupled cells, few and many atom types."""
import numpy as np
import pytest
import torch

from test_adjoint_ref import monoclinic

pytestmark = pytest.mark.gpu

# a term's factors carry about 16 roundings (exponents included) of 2^-24 of its size; with a
# white density gradient the ~400 voxels that count add up to 1 / 20 of the sum of their sizes
TOL = 20 * 16 * 2.0 ** -24


def _grad(coords, dims, typ, rad, ucell, fp64):
    from mdsf import engine
    s = engine.Setup(np.array(coords), dims, typ, rad, 0.3, False, ucell)
    plan = engine.Plan.from_setup(s, fft64=fp64)
    types = torch.from_numpy(s.type_index.astype(np.int32).reshape(-1)).to(plan.device)
    scale = torch.from_numpy(np.ascontiguousarray(s.scale, dtype=np.float64)).to(plan.device)
    c = torch.tensor(coords).to(plan.device)
    gd = torch.from_numpy(np.random.default_rng(5).normal(size=tuple(int(v) for v in s.N)))
    plan.prepare_frame(c[0], types, scale[0], [float(v) for v in s.L], s.arith, s.wrap)
    got = plan.deposit_adjoint(gd).cpu().numpy()
    plan.check_errors()
    plan.close()
    return got


@pytest.mark.parametrize("theta", [None, 120.0])
@pytest.mark.parametrize("n,ncorner,ntypes", [(1, 0, 1), (63, 1, 2), (64, 15, 3), (65, 16, 4),
                                              (128, 17, 5), (200, 33, 20)])
def test_batches(gpu, theta, n, ncorner, ntypes):
    """n atoms within one tile's reach and ncorner at the cell's corner."""
    rng = np.random.default_rng(n)
    box = np.array([24.0, 21.0, 19.5])     # 80 x 70 x 65 -> even sizes, ragged tiles
    inner = box * 0.5 + rng.uniform(-1.0, 1.0, (n, 3))
    edge = rng.uniform(-0.8, 0.8, (ncorner, 3)) % box
    coords = np.concatenate([inner, edge])[None].astype(np.float32)
    names = [f"t{k:02d}" for k in range(min(ntypes, n))]
    rad = {name: (1.0 + k, 0.53 + 0.02 * k) for k, name in enumerate(names)}
    typ = [names[i % len(names)] for i in range(n + ncorner)]
    args = (coords, np.tile(box, (1, 1)), typ, rad, monoclinic(theta))
    got, want = _grad(*args, fp64=False), _grad(*args, fp64=True)
    assert np.abs(got - want).max() <= TOL * np.abs(want).max()
