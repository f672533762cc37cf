"""The batch's per-material reduction at the edges of its rounds of loads
(2,048 tiles a round) and the step state it advances, against each material
alone.

Tolerance: both sides sum fp32 sums of 256 pixels in double and round once;
the pixels' losses may differ by an ulp where a multiply-add is contracted
differently (2^-23 relative on the loss), and each later step starts from
parameters that agree to 1e-5: 1e-5 on the loss."""
import numpy as np
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("light", [False, True])
@pytest.mark.parametrize("sizes", [(725, 16), (724, 257, 1), (1100,)])
def test_losses_and_state_at_the_edges_of_a_round(pkg, sizes, light):
    dev, steps, views = torch.device("cuda:0"), 3, 2
    cam, lpos = (torch.from_numpy(a) for a in pkg.synthetic.flash_grid(n_views=views))

    def problem(res, seed):
        g = torch.Generator().manual_seed(seed)
        r = pkg.Microfacet(res, views, 17.0, [cam, lpos, torch.from_numpy(pkg.synthetic.light_power())], dev)
        target = torch.rand((1, 9, res, res), generator=g) * 0.8 - 0.4
        start = (target + 0.1 * torch.randn(target.shape, generator=g)).to(dev)
        with torch.no_grad():
            photos = r.eval(target.to(dev))
        return r, start, photos

    batch = pkg.BatchedStep([problem(res, i) for i, res in enumerate(sizes)], 0.01, loss="l2", history=steps,
                            config={"tile_pixels": 256, "pixels_per_thread": 1, "views_per_trip": 1,
                                    "blocks_per_cu": -1}, optim_light=light)
    alone = [pkg.FusedStep(*problem(res, i), 0.01, loss="l2", history=steps, optim_light=light)
             for i, res in enumerate(sizes)]
    for _ in range(steps):
        batch.step()
        for f in alone:
            f.step()
    state = batch.read_state()
    assert state["step"] == steps
    assert state["beta1_pow"] == alone[0].read_state()["beta1_pow"]
    hist = batch.loss_history()
    for i, f in enumerate(alone):
        np.testing.assert_allclose(hist[:, i], f.losses(), rtol=1e-5)
