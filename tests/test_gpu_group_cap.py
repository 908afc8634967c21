"""The callers that know their frame count pass it on: plans hold no larger groups than a call can
use, longer calls still work, and S(q) and the gradients keep their bits whatever the group."""
import numpy as np
import pytest
import torch

from test_gpu_frame_groups import CELLS, RAD, _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell,fp64", [("orth", False), ("orth", True), ("xy", False), ("xy", True),
                                       ("general", False)])
def test_results_do_not_depend_on_the_group(gpu, cell, fp64):
    from mdsf import engine
    nframes = 17
    s, plan, coords, types, scale, box = _system(nframes, cell, fp64)
    inside = torch.remainder(coords, torch.tensor(box, device="cuda") * 0.97)
    dsf = torch.randn(plan.half_shape, dtype=torch.float64, device="cuda",
                      generator=torch.Generator("cuda").manual_seed(4))
    want = None
    for cap, group in ((0, 16), (1, 1), (3, 3), (40, 16)):
        p = engine.Plan.from_setup(s, fft64=fp64, max_frames=cap)
        assert p.group == (group, 0)
        p.accumulate_frames(inside.clone(), types, scale, box, s.arith, s.wrap)
        got = [p.sf()]
        if cell != "general":
            got.append(p.adjoint_frames(inside.clone(), types, scale, box, s.arith, s.wrap, dsf))
            assert p.group == (group, group)
        p.check_errors()
        want = want or got
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        p.close()
    plan.close()


def test_callers_pass_their_frames(gpu, tmp_path, monkeypatch):
    import dens
    from mdsf import engine
    from mdsf.autograd import SFModel
    rng = np.random.default_rng(2)
    box, typ = np.array([12.0, 17.0, 14.0]), np.array(["H", "C", "O"] * 20)
    coords = rng.uniform(0, 1, (3, 60, 3)) * box
    dims = np.tile(box, (3, 1))
    model = SFModel(np.array(coords), dims, typ, RAD, 0.6, True, CELLS["orth"])
    assert model.plan.group[0] == 3
    model.close()
    setups = [engine.Setup(np.array(coords[:k]), dims[:k], typ, RAD, 0.6, True, CELLS["orth"])
              for k in (1, 2, 3)]
    batch = engine.Batch(setups)
    assert [p.group[0] for p in batch.plans] == [1, 2, 3]
    # more frames than the setup's: smaller groups, the same sums
    types = torch.from_numpy(setups[0].type_index.astype(np.int32)).cuda()
    sc = torch.ones(3, 3, dtype=torch.float64, device="cuda")
    dev = torch.from_numpy(coords).cuda()
    for i in range(3):
        batch.set_frames(i, dev, types, sc)
    batch.run()
    batch.check_errors()
    assert torch.equal(batch.sf(0), batch.sf(1)) and torch.equal(batch.sf(0), batch.sf(2))
    batch.close()
    made = []
    real = engine.Plan.from_setup.__func__

    def record(cls, s, **kw):
        made.append((kw.get("fft64"), kw.get("max_frames")))
        return real(cls, s, **kw)

    monkeypatch.setattr(engine.Plan, "from_setup", classmethod(record))
    monkeypatch.setattr(dens, "PRINT_DETAILS", False)
    monkeypatch.setattr(dens, "AUTO_FP32_MAX_ERR", 1.0)
    dens.compute_sf(np.array(coords), dims, typ, str(tmp_path / "a"), RAD, CELLS["orth"], 0.6)
    assert made == [(False, 3), (True, 1)]
    made.clear()
    monkeypatch.setattr(dens, "AUTO_FP32_MAX_ERR", -1.0)   # the fallback: an FP64 plan for the run
    monkeypatch.setattr(dens, "CHECKPOINT_FRAMES", 2)
    dens.compute_sf(np.array(coords), dims, typ, str(tmp_path / "b"), RAD, CELLS["orth"], 0.6)
    assert made == [(False, 2), (True, 1), (True, 2)]
