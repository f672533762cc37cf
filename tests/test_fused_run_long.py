"""FusedStep.run past the length from which it replays a recorded stretch: the
bits of one step() per iteration, whatever changes on the way."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("light", [False, True])
def test_recorded_stretches_are_the_step_sequence(pkg, monkeypatch, light):
    for name, value in (("RECORD_AFTER", 8), ("RECORD_STEPS", 3)):
        monkeypatch.setattr(pkg.optim, name, value)
    res, views, dev = 37, 5, torch.device("cuda:0")
    gt = torch.from_numpy(pkg.synthetic.ground_truth_textures(res, seed=0))[None].to(dev)
    cam, lpos = pkg.synthetic.flash_grid(n_views=views)
    start = torch.from_numpy(pkg.synthetic.init_textures(gt[0].cpu().numpy(), seed=1))[None].to(dev)

    def problem():
        power = torch.from_numpy(pkg.synthetic.light_power()).to(dev)
        r = pkg.Microfacet(res, views, 17.0, [torch.from_numpy(cam), torch.from_numpy(lpos), power], dev)
        with torch.no_grad():
            targets = r.eval(gt)
        return pkg.FusedStep(r, start.clone(), targets, 0.01, loss="log_l2", history=80, own_textures=True,
                             optim_light=light)

    a, b = problem(), problem()

    def both(n, run):
        for _ in range(n):
            a.step()
        run()
        assert b.steps_launched == a.steps_launched
        for x, y in ((a.textures, b.textures), (a.exp_avg, b.exp_avg), (a.exp_avg_sq, b.exp_avg_sq),
                     (a.light_pow, b.light_pow)):
            assert torch.equal(x, y)

    both(8, lambda: b.run(8, 4))
    assert b._record is None
    both(14, lambda: b.run(14, 4))          # three recorded pieces and two single launches
    first = b._record
    assert first is not None
    both(8, lambda: b.run(8, 4))
    assert b._record is first
    a.lr = b.lr = 0.003                     # another rate: not the recorded launches
    both(4, lambda: b.run(4, 4))
    both(12, lambda: b.run(12, 4))          # recorded again
    assert b._record is not first
    # recorded by the caller: the launches themselves, every replay the next iterations
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        b.run(4, 4)
    torch.cuda.current_stream().wait_stream(s)
    for k in range(3):
        b.steps_launched = a.steps_launched + 4
        both(4, g.replay)
        torch.cuda.synchronize()
    assert np.array_equal(a.losses(), b.losses()) and len(a.losses()) == a.steps_launched


def test_what_is_not_recorded(pkg, monkeypatch):
    """Short pieces, large maps and short runs launch from the loop."""
    monkeypatch.setattr(pkg.optim, "RECORD_AFTER", 2)
    dev = torch.device("cuda:0")
    cam, lpos = pkg.synthetic.flash_grid(n_views=1)
    for res, per in ((33, pkg.optim.RECORD_STEPS - 1), (pkg.optim.RECORD_RES + 1, pkg.optim.RECORD_STEPS)):
        power = torch.from_numpy(pkg.synthetic.light_power()).to(dev)
        r = pkg.Microfacet(res, 1, 17.0, [torch.from_numpy(cam), torch.from_numpy(lpos), power], dev)
        f = pkg.FusedStep(r, torch.zeros((1, 9, res, res), device=dev), torch.full((1, 3, res, res), 0.5, device=dev),
                          0.01)
        f.run(3 * per, per)
        assert f._record is None and f.steps_launched == 3 * per
