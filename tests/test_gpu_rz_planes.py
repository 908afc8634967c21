"""The separable form of the cylindrical average (z axis orthogonal to x and y) at the edges of
its rounds -- z planes, staged samples, z bins off the grid's own -- against the mean of the
pointwise interpolant over the same samples (plot2d.py:605-627)."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# a mean of up to 1,500 positive samples, each a sum of 8 products: either order of the additions
# is within (1500 + 16) eps of the exact value, the two within twice that
RTOL = 2 * 1516 * 2.0 ** -53


def _average(kp, rarr, nth, zar, binv):
    from mdsf import _lib
    lib = _lib.load()
    nx, ny, nz = kp.shape[:3]
    r, z = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in (rarr, zar))
    n = torch.tensor(nth, dtype=torch.int32, device="cuda")
    oa = torch.empty(len(rarr), len(zar), dtype=torch.float64, device="cuda")
    p = _lib.c_void_p
    b = np.ascontiguousarray(binv)
    _lib.check(lib.mdsf_rz_average(p(kp.data_ptr()), nx, ny, nz, p(r.data_ptr()), p(n.data_ptr()),
                                   len(rarr), p(z.data_ptr()), len(zar),
                                   b.ctypes.data_as(_lib.ctypes.POINTER(_lib.c_double)),
                                   p(oa.data_ptr()), p(torch.cuda.current_stream().cuda_stream)))
    return oa


@pytest.mark.parametrize("n,nzb,nth", [
    ((6, 5, 2), 3, [1, 2, 3]),
    ((9, 12, 255), 255, [1, 5, 64]),
    ((8, 7, 256), 300, [3, 1023, 1024]),
    ((7, 9, 257), 64, [1025, 4, 1500]),
    ((5, 6, 1024), 17, [7, 1, 2]),
    ((5, 6, 1025), 17, [7, 1, 2]),      # past the plane sums in LDS: the general form
])
@pytest.mark.parametrize("theta", [90, 120])
def test_rz_average_matches_pointwise_mean(gpu, n, nzb, nth, theta):
    from mdsf import engine
    g = torch.Generator().manual_seed(sum(n))
    ax = [torch.linspace(-1.0 - 0.1 * d, 1.3 + 0.2 * d, m, dtype=torch.float64)
          for d, m in enumerate(n)]
    kp = torch.stack(torch.meshgrid(*ax, indexing="ij")
                     + (torch.rand(n, dtype=torch.float64, generator=g) + 0.25,), -1).cuda()
    t = math.radians(theta)
    binv = np.array([[1.0, 0, 0], [math.cos(t) if theta != 90 else 0.0, math.sin(t), 0], [0, 0, 1]])
    rarr = [0.0, 0.6, 0.8][:len(nth)]
    # one z past the grid: a NaN column
    zar = np.concatenate([np.linspace(float(ax[2][0]), float(ax[2][-1]), nzb - 1),
                          [float(ax[2][-1]) + 0.1]])
    got = _average(kp, rarr, nth, zar, binv)
    b = torch.from_numpy(binv).cuda()
    for i, (r, m) in enumerate(zip(rarr, nth)):
        th = torch.arange(m, dtype=torch.float64, device="cuda") * (2 * math.pi / m)
        p = torch.empty(m, nzb, 3, dtype=torch.float64, device="cuda")
        p[..., 0], p[..., 1] = (r * th.cos())[:, None], (r * th.sin())[:, None]
        p[..., 2] = torch.from_numpy(zar).cuda()
        want = engine.interp_points(kp, (p.reshape(-1, 3) @ b).reshape(m, nzb, 3)).mean(0)
        assert bool(torch.isnan(got[i, -1])) and bool(torch.isnan(want[-1]))
        # the sample points of the two forms agree to a few ulp, their values to the local slope
        torch.testing.assert_close(got[i, :-1], want[:-1], rtol=RTOL, atol=200 * 2.0 ** -53)


@pytest.mark.parametrize("nz", [3, 8, 9, 10, 12, 17, 18])
def test_rz_average_of_few_planes(gpu, nz):
    """Bands of z cells that are empty, of one cell, or short at the end."""
    test_rz_average_matches_pointwise_mean(gpu, (6, 7, nz), 2 * nz + 1, [1, 600, 37], 120)


def test_rz_average_ring_off_the_grid_is_nan(gpu):
    ax = [torch.linspace(-1, 1, m, dtype=torch.float64) for m in (5, 6, 7)]
    kp = torch.stack(torch.meshgrid(*ax, indexing="ij") + (torch.ones(5, 6, 7, dtype=torch.float64),),
                     -1).cuda()
    got = _average(kp, [0.5, 1.2], [8, 8], [-0.5, 0.0, 0.5], np.eye(3))
    torch.testing.assert_close(got[0], torch.ones(3, dtype=torch.float64, device="cuda"), rtol=1e-14,
                               atol=0)
    assert bool(torch.isnan(got[1]).all())


@pytest.mark.parametrize("nr,nzb", [(1, 1), (1, 300), (3, 255), (257, 64), (400, 257)])
@pytest.mark.parametrize("nans", ["none", "some", "all"])
@pytest.mark.parametrize("normalise", [0, 1])
def test_rz_finish(gpu, nr, nzb, nans, normalise):
    """NaN bins, mean and mirror (plot2d.py:629-637) against torch's operations."""
    from mdsf import _lib
    g = torch.Generator().manual_seed(nr + nzb)
    oa = torch.rand(nr, nzb, dtype=torch.float64, generator=g) + 0.25
    if nans == "all":
        oa[:] = float("nan")
    elif nans == "some":
        oa[torch.rand(nr, nzb, generator=g) < 0.3] = float("nan")
    bad = torch.isnan(oa)
    low = oa[~bad].min() if bool((~bad).any()) else torch.tensor(float("nan"), dtype=torch.float64)
    want = torch.where(bad, low, oa)
    if normalise:
        want = want / want.mean()
    d = oa.cuda()
    fin = torch.empty(2 * nr - 1, nzb, dtype=torch.float64, device="cuda")
    work = torch.empty(3 * nr, dtype=torch.float64, device="cuda")
    p = _lib.c_void_p
    _lib.check(_lib.load().mdsf_rz_finish(p(d.data_ptr()), nr, nzb, normalise, p(fin.data_ptr()),
                                          p(work.data_ptr()),
                                          p(torch.cuda.current_stream().cuda_stream)))
    # the mean: sums of positive values in two orders
    tol = 2 * (nr * nzb) ** 0.5 * 2.0 ** -53 * 8
    torch.testing.assert_close(d.cpu(), want, rtol=tol, atol=0, equal_nan=True)
    mirrored = torch.cat([torch.flip(d, [0]), d[1:]], 0)
    torch.testing.assert_close(fin, mirrored, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("n", [(2, 4, 6), (4, 2, 6), (4, 6, 2), (6, 4, 64), (4, 4, 66), (8, 10, 130)])
@pytest.mark.parametrize("f32", [False, True])
def test_output_grids(gpu, n, f32):
    """sfplt, kgrid and kgridplt (dens.py:323-344) against the oracle, each alone as well, into
    buffers that are aligned to 8 bytes only."""
    from mdsf import _lib, engine
    from oracle import dens_oracle as O
    nx, ny, nz = n
    L = np.array([4.5, 5.25, 6.125], dtype=np.float32 if f32 else np.float64)
    sf = np.random.default_rng(sum(n)).random((nx, ny, nz // 2 + 1)) + 0.5
    # an axis of two points leaves no plot grid
    splt = O.get_dplot(sf) if min(nx, ny) > 2 else np.zeros((nx - 2, ny - 2, nz - 1))
    if nz == 2 and splt.size:
        # the mean in the centre reads a plane that get_dplot leaves as np.empty made it
        splt[splt.shape[0] // 2, splt.shape[1] // 2, 0] = (sf[1, 0, 0] + sf[0, 1, 0]
                                                           + sf[0, 0, 1]) * (1.0 / 3.0)
    kg, kgp = O.kgrids(sf.shape, L, splt)
    plan = engine.Plan(list(n), 0, [1.0] * 3, np.eye(3), [], [], [], [])
    p = _lib.c_void_p
    d_sf = torch.from_numpy(sf).cuda()

    def run(which):
        sizes = [splt.size, sf.size * 4, kgp.size]
        bufs = [torch.full((m + 2,), -7.0, dtype=torch.float64, device="cuda") for m in sizes]
        ptr = [p(b.data_ptr() + 8) if w else p(0) for b, w in zip(bufs, which)]
        _lib.check(_lib.load().mdsf_outputs(plan._handle, p(d_sf.data_ptr()),
                                            _lib.doubles([float(x) for x in L]), int(f32), *ptr,
                                            p(torch.cuda.current_stream().cuda_stream)))
        out = [b.cpu().numpy() for b in bufs]
        for o, m, w in zip(out, sizes, which):
            assert o[0] == -7.0 and o[m + 1] == -7.0
        return [o[1:-1] for o in out]

    all3 = run((1, 1, 1))
    assert np.array_equal(all3[0], splt.ravel())
    assert np.array_equal(all3[1], kg.ravel())
    assert np.array_equal(all3[2], kgp.ravel())
    for k in range(3):
        alone = run([j == k for j in range(3)])
        for j in range(3):
            assert np.array_equal(alone[j], all3[j] if j == k else np.full_like(all3[j], -7.0))
    plan.close()
