"""FP64 plans of general cells (z coupled to x and y) evaluate one exponential per voxel (dens.py:301-308):
a voxel's value depends on its offset from the atom alone, so an atom moved by whole cells leaves the
same bits, wherever its window falls in the tiles, and every value is within the roundings of one
exponential of the exact one, at fine resolution too."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CELLS = {"dodecahedron": np.array([[1.0, 0, 0], [0.5, np.sqrt(0.75), 0],
                                   [0.5, np.sqrt(3.0) / 6, np.sqrt(2.0 / 3)]]),
         "oblique": np.array([[1.0, 0, 0], [0, 1, 0], [-0.6, 0.5, 0.62]])}


@pytest.mark.parametrize("cell", list(CELLS))
@pytest.mark.parametrize("name,sres,n", [("O", 0.25, 64), ("C", 0.25, 72), ("H", 0.5, 40), ("O", 0.5, 42),
                                         ("C", 1.0, 36)])
def test_values_follow_the_atom(gpu, rad, name, sres, n, cell):
    from mdsf import engine
    ucell, dr = CELLS[cell], sres
    rng = np.random.default_rng(n)
    # offsets and cell edges that are exact in binary, a window off the cell's faces
    r = (n // 2 - 7) * dr + np.floor(rng.uniform(0, dr, 3) * 1024) / 1024
    coords = r[None, None, :]
    s = engine.Setup(np.array(coords), np.full((1, 3), n * dr), [name], rad, sres, False, ucell)
    assert list(s.N) == [n] * 3 and float(s.dr[0]) == dr
    half = [int(h) for h in s.half[0]]
    plan = engine.Plan.from_setup(s, fft64=True)
    types = torch.from_numpy(s.type_index.astype(np.int32)).cuda()
    scale = torch.from_numpy(np.ascontiguousarray(s.scale)).cuda()

    def density(shift):
        c = torch.from_numpy(r + np.array(shift) * dr)[None].cuda()
        return plan.deposit_fold(c, types, scale, [float(x) for x in s.L], s.arith, s.wrap)

    first = density((0, 0, 0))
    plan.check_errors()
    for k in range(1, 15):
        moved = density((k % 5, 2 * (k % 4), k))
        assert torch.equal(moved, torch.roll(first, (k % 5, 2 * (k % 4), k), (0, 1, 2))), k
    # against extended precision: the exponent's terms carry up to 10 roundings each, the
    # exponential and the amplitude 6
    q = np.longdouble
    G = (ucell @ ucell.T).astype(q)
    home = [int(r[d] / dr) for d in range(3)]
    b = [q(r[d]) - np.arange(home[d] - half[d], home[d] + half[d]).astype(q) * q(dr) for d in range(3)]
    bx, by, bz = b[0][:, None, None], b[1][None, :, None], b[2][None, None, :]
    terms = [G[0, 0] * bx * bx, G[1, 1] * by * by, G[2, 2] * bz * bz, 2 * G[0, 1] * bx * by,
             2 * G[0, 2] * bx * bz, 2 * G[1, 2] * by * bz]
    nel, sigma = rad[name]
    k2 = q(1) / q(2 * np.power(sigma, 2.0))
    want = q(nel / np.power(sigma, 3.0)) * np.exp(-sum(terms) * k2)
    size = sum(np.abs(t) for t in terms) * k2
    got = first.cpu().numpy()[tuple(slice(home[d] - half[d], home[d] + half[d]) for d in range(3))]
    assert np.all(np.abs(got - want) <= (10 * size + 6) * q(2.0) ** -53 * want)
    plan.close()
