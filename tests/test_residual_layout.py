"""The y pass's 4-bit residuals on their way to the x pass (FP32 plans, dens.py:313-318), in every
layout: blocks of x next to powers of two, rows elsewhere.

The density lies in the plane z = 0: its z transform is the density itself, exact in FP32, and the x
pass sums |F|^2 in FP64, so what the y pass stores is the only rounding left.  A stored component y
is off by at most half a sixteenth of an ulp (an ulp at the top of the residual's range), about
2^-27 |y| / sqrt(12) rms or less, the x pass adds nx of them, and the error of S along F is
  e = (S - |F|^2) / 2 |F|,  rms <= sqrt(nx) 2^-27 sigma / sqrt(12),  sigma^2 = ny var / 2.
Without residuals, or with any other value's, e is 16 times that and more; the bound is twice it."""
import numpy as np
import pytest

SHAPES = [(16, 16), (16, 512), (512, 16), (64, 1024), (1024, 64), (32, 256), (256, 128), (512, 512),
          (1024, 1024), (64, 90), (90, 64), (128, 32), (64, 64)]
BOUND = 2.0


def plane(nx, ny):
    return (np.random.default_rng(nx * 2048 + ny).random((nx, ny)) - 0.5).astype(np.float32)


def statistic(sf, d):
    """rms of e in units of the bound's sqrt(nx) 2^-27 sigma / sqrt(12), for S(q) of the half kz = 0."""
    nx, ny = d.shape
    F = np.abs(np.fft.fft2(d.astype(np.float64)))
    e = (sf - F * F) / (2 * F)
    keep = F > 0.1 * np.sqrt(np.mean(F * F))       # no division by bins that happen to be faint
    sigma = np.sqrt(ny * np.mean(d.astype(np.float64) ** 2) / 2)
    return np.sqrt(np.mean(e[keep] ** 2)) / (np.sqrt(nx) * 2.0 ** -27 * sigma / np.sqrt(12))


@pytest.mark.parametrize("nx,ny", [(64, 64), (16, 512), (512, 128)])
def test_the_statistic_tells_residuals_apart(nx, ny):
    """On the host: correct residuals pass by far, missing, negated and misplaced ones fail by far."""
    d = plane(nx, ny)
    y = np.fft.fft(d.astype(np.float64), axis=1)
    parts = np.stack([y.real, y.imag])
    h = parts.astype(np.float32)
    ulp = np.spacing(np.abs(h)).astype(np.float64)
    r = np.clip(np.rint((parts - h) * 16 / ulp), -8, 7)
    rng = np.random.default_rng(1)
    for name, res in (("correct", r), ("none", 0 * r), ("negated", -r),
                      ("shifted", np.roll(r, 1, axis=1)), ("other", rng.permutation(r.ravel()).reshape(r.shape))):
        v = h + res * ulp / 16
        F = np.fft.fft(v[0] + 1j * v[1], axis=0)
        s = statistic(np.abs(F) ** 2, d)
        assert s < BOUND / 2 if name == "correct" else s > 4 * BOUND, (name, s)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", SHAPES)
def test_plans_pass_the_residuals_on(gpu, nx, ny):
    import torch

    from mdsf import engine
    d = plane(nx, ny)
    nz = 8
    density = torch.zeros(nx, ny, nz, dtype=torch.float32)
    density[:, :, 0] = torch.from_numpy(d)
    plan = engine.Plan((nx, ny, nz), 0, [1.0] * 3, np.eye(3), [], [], [], [])
    plan.reset()
    plan.accumulate_density(density)
    sf = plan.sf().cpu().numpy()
    plan.close()
    for kz in range(nz // 2):
        assert statistic(sf[:, :, kz], d) < BOUND, kz
    # the Nyquist plane stays in FP64
    assert statistic(sf[:, :, nz // 2], d) < 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(64, 32, 32), (32, 128, 32), (128, 64, 32), (16, 256, 32), (32, 32, 64)])
def test_groups_and_pairs_of_frames(gpu, n):
    """Frames side by side in a group, and x passes of two frames in one launch, read each frame's own
    residuals: the same bits as frame by frame."""
    import torch

    from mdsf import engine
    rng = np.random.default_rng(n[0])
    box = np.array(n) * 0.5
    typ, frames = ["H", "C", "O"] * 40, 7
    coords = rng.uniform(0, 1, (frames, 120, 3)) * box
    rad = {"H": (1.0, 0.35), "C": (6.0, 0.4), "O": (8.0, 0.45)}
    s = engine.Setup(np.array(coords), np.tile(box, (frames, 1)), typ, rad, 0.5, False, np.eye(3))
    assert tuple(s.N) == n
    types = torch.from_numpy(s.type_index.astype(np.int32)).cuda()
    scale = torch.from_numpy(np.ascontiguousarray(s.scale)).cuda()
    dev = torch.from_numpy(coords).cuda()
    sums = []
    for cap, step in ((0, frames), (1, frames), (2, frames), (1, 1)):   # one group, pairs, groups of 2
        plan = engine.Plan.from_setup(s, max_frames=cap)
        plan.reset()
        for t in range(0, frames, step):
            plan.accumulate_frames(dev[t:t + step].clone(), types, scale[t:t + step],
                                   [float(x) for x in s.L], s.arith, s.wrap)
        plan.check_errors()
        sums.append(plan.sf())
        plan.close()
    assert float(sums[0].max()) > 0
    assert all(torch.equal(a, sums[-1]) for a in sums)
