"""FusedStep.run: the library's own launch loop (svbrdf_fused_steps) against
one step() call per iteration, bit for bit, also when a caller records it."""
import ctypes

import numpy as np
import pytest
import torch


def test_fused_steps_refuses_a_negative_count(pkg):
    lib, f = pkg._lib.load(), ctypes.c_void_p(0x10000)
    args = (f, f, f, f, 64, 0, 0, 9, 17.0, f, f, f, 0, 0, 0.01, 0.9, 0.999, 1e-8, f, None, 0, f, 1 << 30, None)
    assert lib.svbrdf_fused_steps(-1, *args) == -1
    assert lib.svbrdf_fused_steps(0, *args) == 0       # nothing to launch
    bad = list(args)
    bad[4] = 0                                          # the step's own checks
    assert lib.svbrdf_fused_steps(1, *bad) == -2


@pytest.mark.gpu
@pytest.mark.parametrize("light", [False, True])
@pytest.mark.parametrize("n,graph_steps", [(1, 100), (7, 3), (12, 12)])
def test_run_is_the_step_sequence(pkg, n, graph_steps, light):
    res, views, dev = 37, 5, torch.device("cuda:0")
    gt = torch.from_numpy(pkg.synthetic.ground_truth_textures(res, seed=0))[None].to(dev)
    cam, lpos = pkg.synthetic.flash_grid(n_views=views)
    start = torch.from_numpy(pkg.synthetic.init_textures(gt[0].cpu().numpy(), seed=1))[None].to(dev)

    def problem():
        power = torch.from_numpy(pkg.synthetic.light_power()).to(dev)
        r = pkg.Microfacet(res, views, 17.0, [torch.from_numpy(cam), torch.from_numpy(lpos), power], dev)
        with torch.no_grad():
            targets = r.eval(gt)
        return pkg.FusedStep(r, start.clone(), targets, 0.01, loss="log_l2", history=2 * n, own_textures=True,
                             optim_light=light)

    a, b = problem(), problem()
    for _ in range(2 * n):
        a.step()
    b.run(n, graph_steps)
    g = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        b.run(n, graph_steps)
    torch.cuda.current_stream().wait_stream(s)
    g.replay()
    assert b.steps_launched == 2 * n
    for x, y in ((a.textures, b.textures), (a.exp_avg, b.exp_avg), (a.exp_avg_sq, b.exp_avg_sq),
                 (a.light_pow, b.light_pow)):
        assert torch.equal(x, y)
    assert np.array_equal(a.losses(), b.losses()) and len(a.losses()) == 2 * n
