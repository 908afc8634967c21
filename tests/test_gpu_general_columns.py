"""The column form of the general-cell deposition against the full sum over windows (dens.py:283-311)
where its conditions change: corner atoms, windows as wide as the grid (two images in a tile), last
tiles of 2 to 16 cells, and a cell matrix far from unit edges (factors beyond FP64's range)."""
import numpy as np
import pytest
import torch

from oracle import dens_oracle as O

pytestmark = pytest.mark.gpu

DODECAHEDRON = np.array([[1.0, 0, 0], [0.5, np.sqrt(0.75), 0], [0.5, np.sqrt(3.0) / 6, np.sqrt(2.0 / 3)]])
CELLS = {"dodecahedron": DODECAHEDRON, "oblique": np.array([[1.0, 0, 0], [0, 1, 0], [-0.6, 0.5, 0.62]]),
         "long edges": 30.0 * DODECAHEDRON}


# (FP64 with long edges is left out: b^T G b cancels there, and the last bits of its terms, which the
# oracle adds in another order, are worth more than the bound below)
@pytest.mark.parametrize("cell,fp64", [("dodecahedron", False), ("dodecahedron", True),
                                       ("oblique", False), ("oblique", True), ("long edges", False)])
@pytest.mark.parametrize("box,sres", [((12.0, 12.6, 13.0), 0.7), ((24.5, 20.0, 25.2), 0.5)])
def test_density(gpu, rad, box, sres, cell, fp64):
    from mdsf import engine
    rng = np.random.default_rng(7)
    L, natoms = np.array(box), 70
    typ = [("H", "C", "O")[k % 3] for k in range(natoms)]
    coords = (rng.uniform(0.0, 1.0, size=(1, natoms, 3)) * L)
    coords[0, :12] = np.mod(rng.normal(0.0, 0.7, size=(12, 3)), L)
    dims, ucell = np.tile(L, (1, 1)), CELLS[cell]
    s = engine.Setup(np.array(coords), dims, typ, rad, sres, True, ucell)
    o = O.setup(np.array(coords), np.array(dims), typ, rad, sres, better=True)
    n, nb = o["N"], o["Nb"]
    d0, _ = O.deposit_frame(coords[0], list(typ), rad, o["bdict"], o["dr"], nb, ucell,
                            tuple(int(n[i]) + 2 * nb for i in range(3)))
    want = O.fold(d0, *O.fold_tables(n, nb))
    plan = engine.Plan.from_setup(s, fft64=fp64)
    got = plan.deposit_fold(torch.from_numpy(coords[0]).cuda(),
                            torch.from_numpy(s.type_index.astype(np.int32)).cuda(),
                            torch.from_numpy(np.ascontiguousarray(s.scale)).cuda(),
                            [float(x) for x in s.L], s.arith, s.wrap)
    plan.check_errors()
    # exponents up to 55 (and their rounding) plus a few products per term; FP32: one rounding, and
    # FP32 exponentials in the corner spill
    tol = 200 * 2.0 ** -53 if fp64 else 2e-6
    np.testing.assert_allclose(got.cpu().numpy(), want, rtol=tol, atol=tol * want.max())
    plan.close()
