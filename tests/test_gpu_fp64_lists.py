"""FP64 deposition from the tile lists at the edges of its batches (64 regular atoms, 16 corner atoms)
and of its tiles (grids that 16 does not divide), against the FP64 oracle (dens.py:283-311)."""
import numpy as np
import pytest
import torch

from oracle import dens_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms", [1, 63, 64, 65, 193])
@pytest.mark.parametrize("box", [(16.0, 17.0, 18.0), (30.0, 24.0, 33.0)])
def test_density(gpu, rad, natoms, box):
    from mdsf import engine
    rng = np.random.default_rng(natoms)
    L = np.array(box)
    typ = [("H", "C", "O")[k % 3] for k in range(natoms)]
    # everything within one tile's reach, and as many corner atoms as fill two batches
    coords = (rng.uniform(0.0, 1.0, size=(1, natoms, 3)) * 6.0).astype(np.float64)
    ncorner = min(natoms // 2, 33)
    coords[0, :ncorner] = np.mod(rng.normal(0.0, 0.4, size=(ncorner, 3)), L)
    dims = np.tile(L, (1, 1))
    s = engine.Setup(np.array(coords), dims, typ, rad, 0.7, True, np.eye(3))
    o = O.setup(np.array(coords), np.array(dims), typ, rad, 0.7, better=True)
    n, nb = o["N"], o["Nb"]
    d0, _ = O.deposit_frame(coords[0], list(typ), rad, o["bdict"], o["dr"], nb, np.eye(3),
                            tuple(int(n[i]) + 2 * nb for i in range(3)))
    want = O.fold(d0, *O.fold_tables(n, nb))
    plan = engine.Plan.from_setup(s, fft64=True)
    types = torch.from_numpy(s.type_index.astype(np.int32)).cuda()
    scale = torch.from_numpy(np.ascontiguousarray(s.scale)).cuda()
    got = plan.deposit_fold(torch.from_numpy(coords[0]).cuda(), types, scale,
                            [float(x) for x in s.L], s.arith, s.wrap)
    plan.check_errors()
    # products of three factors of a few ulp each, summed over at most natoms terms
    tol = (16 + natoms) * 2.0 ** -53
    np.testing.assert_allclose(got.cpu().numpy(), want, rtol=tol, atol=tol * want.max())
    plan.close()
