"""The denoiser's kernels at sizes that their tiles do not divide (tiles of
32 x 8 pixels, strips of 32 rows), against the FP64 evaluation of
oracle/denoise_oracle.py, with the bars of test_gpu_denoise.py."""
import numpy as np
import pytest

import denoise_oracle as orc
from test_gpu_denoise import BLOCKS, relnorm

pytestmark = pytest.mark.gpu

SIZES = [(5, 32), (9, 32), (31, 64), (33, 32), (70, 96)]


def case(zp, H, W, scale=0.3):
    rng = np.random.default_rng(H * 1000 + W)
    dn = zp.Denoiser(H, W)
    dn.set_scale(scale)
    p = dn.params().astype(np.float64)
    for off, n in ((1200, 16), (7616, 16), (8832, 3)):
        p[off:off + n] = rng.normal(0, 0.1, n)
    dn.set_params(p)
    x = rng.normal(0, scale, (H, W, 3)).astype(np.float32)
    t = (0.5 * x + rng.normal(0, 0.1 * scale, (H, W, 3))).astype(np.float32)
    return dn, p, x, t, scale


@pytest.mark.parametrize("H,W", SIZES)
def test_forward_and_gradient(H, W):
    import pyzpic as zp
    dn, p, x, t, scale = case(zp, H, W)
    assert relnorm(dn.forward(x), orc.forward(p, x, scale, bf=True)["out"]) <= 5e-3
    loss, g = dn.gradient(x, t)
    ref_loss, ref_g = orc.loss_and_grad(p, x, t, scale, bf=True)
    assert abs(loss - ref_loss) <= 1e-2 * ref_loss
    for name, a, b in BLOCKS:
        assert relnorm(g[a:b], ref_g[a:b]) <= 3e-2, name
    dn.close()


@pytest.mark.parametrize("H,W", [(9, 32), (40, 64)])
def test_training_moves_weights_and_operands_alike(H, W):
    """After some steps the network of the moved operands is that of the
    parameters it reports, and the losses are those of single evaluations."""
    import pyzpic as zp
    dn, p, x, t, scale = case(zp, H, W)
    train = zp.Denoiser(H, W, 2, params=p.astype(np.float32), scale=scale)
    sims = [zp.Simulation((W // 32, 1), (32, H), (W * 0.1, H * 0.1), 0.05) for _ in range(2)]
    g = sims[0].geom
    for sim, f in zip(sims, (x, t)):
        J = np.zeros((sim.ntiles, g.tile_vol, 3), np.float32)
        view = J[:, :g.ext_x * g.ext_y].reshape(sim.ntiles, g.ext_y, g.ext_x, 3)
        view[:, 1:1 + H, 1:33] = f.reshape(H, W // 32, 32, 3).transpose(1, 0, 2, 3)
        sim.set_field("J", J)
    sims[0].add_pair_to(train, sims[1])
    losses = train.train(3, lr=1e-3, seed=1)
    assert losses[0] == pytest.approx(dn.gradient(x, t)[0], rel=1e-12)
    assert losses[2] < losses[0]
    dn.set_params(train.params())
    assert np.array_equal(train.forward(x), dn.forward(x))
    assert not np.array_equal(train.params(), p.astype(np.float32))
    for sim in sims:
        sim.close()
