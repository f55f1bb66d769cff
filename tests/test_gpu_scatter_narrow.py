"""Fields of at most 8 channels take the direct scatter for few rows and the sorted
one from 98,304: the factor gradients of a render on both sides of that line, and of
tiny ones, are the float64 sums of those of parts (2e-4 of the largest: the order of
the FP32 sums), for both fields, all samples shaded or some; and a small training
step of such fields sorts nothing."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, mlp_module, oracle_params, report, to_device_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cd,ca", [(1, 7), (4, 8), (8, 24), (8, 18), (16, 8)])
@pytest.mark.parametrize("rays,n,k", [(3, 17, 17), (511, 192, 192), (512, 192, 192), (511, 192, 30),
                                      (512, 192, 30), (3300, 40, 30)])
def test_factor_gradients(rays, n, k, cd, ca):
    log(f"case: {rays} rays x {n} samples, {k} shaded, {cd} and {ca} channels")
    from tensorf_amd import cameras, render
    shape = orc.MlpShape(feat_dim=3 * ca)
    p = oracle_params(24, cd, ca, shape, seed=5, std=0.3, bias_std=0.1)
    den, app, mp = to_device_params(p, shape)
    lp = render.LearnableParams(mp, app, den, False)
    o, d = orc.make_rays(rays, seed=4, radius=3.0, target_half=0.6)
    batch = cameras.Rays3D(dev(f32(o)), dev(f32(d)),
                           torch.zeros(rays, dtype=torch.int32, device="cuda"))
    box = dev(np.array([[-1.5] * 3, [1.5] * 3]))
    cfg = render.RenderConfig(0.05, 200.0, render.RenderMode.RGB, n, k, density_shift=0.0)
    mlp = mlp_module(shape)
    leaves = [t.requires_grad_(True) for t in render._leaves(lp)[:4]]
    up = torch.randn(rays, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(1))

    def gradients(a, b):
        out = render.render_rays(mlp, lp, box, batch.slice(a, b), 3, cfg)
        return torch.autograd.grad(out, leaves, up[a:b])

    whole = gradients(0, rays)
    sums = [torch.zeros_like(t, dtype=torch.float64) for t in leaves]
    part = max(1, rays // 2)
    for at in range(0, rays, part):
        for s, g in zip(sums, gradients(at, min(at + part, rays))):
            s += g.double()
    names = ["density plane", "density line", "appearance plane", "appearance line"]
    for name, g, s in zip(names, whole, sums):
        e = report(name, g.cpu().numpy(), s.cpu().numpy())
        assert e.max() <= 2e-4 * float(s.abs().max()), name


@pytest.mark.parametrize("rays,n,k", [(64, 32, 32), (64, 128, 32)])
def test_few_rows_are_not_sorted(rays, n, k):
    """The stages of a small step of narrow fields hold no sort."""
    from tensorf_amd import _lib, cameras, training
    cfg = training.TensorfConfig(
        minibatch_size=rays, n_iters=100, initial_aabb_min=(-1.5,) * 3,
        initial_aabb_max=(1.5,) * 3, appearance_feat_dim=8, density_feat_dim=4, feature_n_freqs=2,
        viewdir_n_freqs=2, grid_dim_init=24, grid_dim_final=24, upsamp_iters=(),
        density_samples_per_ray=n, appearance_samples_per_ray=k)
    st = training.TrainState.initialize(cfg, 24, prng_key=3, num_cameras=1)
    o, d = orc.make_rays(rays, seed=8, radius=4.0, target_half=0.5)
    batch = cameras.RenderedRays(torch.full((rays, 3), 0.5, device="cuda"), cameras.Rays3D(
        dev(f32(o)), dev(f32(d)), torch.zeros(rays, dtype=torch.int32, device="cuda")))
    st.training_step(batch)
    torch.cuda.synchronize()
    _lib.profile_enable(True)
    st.training_step(batch)
    torch.cuda.synchronize()
    stages = _lib.profile_read()
    _lib.profile_enable(False)
    log(f"  stages: {sorted(stages)}")
    assert "adam" in stages and not any("sort" in s for s in stages)
