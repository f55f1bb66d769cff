"""Factor gradients of the render backward over the channel counts and sampling
densities that choose between the scatter's walks: 16 lanes of four channels,
16 or 8 lanes of one, and the general passes (more than 16 channels, not a
multiple of 4); both fields in one walk, or each its own (top-k); line cells in
ray order or (few samples for the grid) sorted. Against the float64 oracle,
2e-4 of the largest gradient (the order of the FP32 sums), as in the other
gradient tests."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, mlp_module, oracle_params, report, to_device_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("contraction", [False, True])
@pytest.mark.parametrize("n,k", [(41, 41), (41, 7), (9, 9), (9, 4), (7, 7)])
@pytest.mark.parametrize("cd,ca", [(8, 24), (5, 20), (1, 17), (16, 48), (13, 64), (24, 8),
                                   (18, 16)])
def test_factor_gradients(cd, ca, n, k, contraction):
    log(f"case: {cd} / {ca} channels, {n} samples, {k} shaded, contraction {contraction}")
    from tensorf_amd import cameras, networks, render
    g, r = 12, 37
    shape = orc.MlpShape(feat_dim=3 * ca)
    p = oracle_params(g, cd, ca, shape, seed=5, std=0.4, bias_std=0.1)
    den, app, mp = to_device_params(p, shape)
    lp = render.LearnableParams(mp, app, den, contraction)
    ds, as_ = den.stacked_single_vm, app.stacked_single_vm
    leaves = [ds.plane, ds.line, as_.plane, as_.line, *networks.FeatureMlp.flat_leaves(mp)]
    for t in leaves:
        t.requires_grad_(True)
    o, d = orc.make_rays(r, seed=4, radius=3.0, target_half=1.2)  # some rays leave by the edges
    o, d = f32(o), f32(d)
    box = np.array([[-1.5] * 3, [1.5] * 3]) * (4.0 / 3.0 if contraction else 1.0)
    rays = cameras.Rays3D(dev(o), dev(d), torch.zeros(r, dtype=torch.int32, device="cuda"))
    cfg = render.RenderConfig(0.05, 200.0, render.RenderMode.RGB, n, k, density_shift=0.0)
    out = render.render_rays(mlp_module(shape), lp, dev(box), rays, 3, cfg)
    up = f32(np.random.default_rng(6).normal(size=(r, 3)))
    (out * dev(up)).sum().backward()
    jit = render.uniform(render._seed(3, 1), r * n if contraction else n).cpu().numpy()
    jit = jit.astype(np.float64).reshape((r, n) if contraction else (n,))
    ocfg = orc.RenderConfig(0.05, 200.0, orc.RGB, n, k, contraction, density_shift=0.0)
    _, cache = orc.render_rays(p, box, o, d, np.zeros(r), ocfg, shape, jit)
    want = orc.render_rays_backward(p, cache, up, ocfg, shape)
    got = {"density_matrix": ds.plane.grad.permute(0, 3, 1, 2),
           "density_vector": ds.line.grad.permute(0, 2, 1),
           "appearance_matrix": as_.plane.grad.permute(0, 3, 1, 2),
           "appearance_vector": as_.line.grad.permute(0, 2, 1)}
    for name, t in got.items():
        e = report(f"grad {name}", t.cpu().numpy(), want[name])
        assert e.max() <= 2e-4 * np.abs(want[name]).max() + 1e-7, name


@pytest.mark.parametrize("k", [48, 5])
@pytest.mark.parametrize("r", [2500, 4000, 8192])
def test_long_walks_match_the_sum_of_short_ones(r, k):
    """A walk takes 8 pairs where there are few and up to 64 where there are many
    (3 * r * 48 pairs here: 16, 32 and 64). The gradient of one call is the sum
    of the gradients of its parts, whose walks are all of 8."""
    log(f"case: {r} rays, {k} shaded")
    from tensorf_amd import cameras, networks, render
    g, n, cd, ca, part = 24, 48, 8, 24, 512
    shape = orc.MlpShape(feat_dim=3 * ca)
    p = oracle_params(g, cd, ca, shape, seed=5, std=0.4, bias_std=0.1)
    den, app, mp = to_device_params(p, shape)
    lp = render.LearnableParams(mp, app, den, False)
    leaves = [den.stacked_single_vm.plane, den.stacked_single_vm.line,
              app.stacked_single_vm.plane, app.stacked_single_vm.line]
    for t in [*leaves, *networks.FeatureMlp.flat_leaves(mp)]:
        t.requires_grad_(True)
    o, d = orc.make_rays(r, seed=4, radius=3.0, target_half=1.2)
    o, d = dev(f32(o)), dev(f32(d))
    up = dev(f32(np.random.default_rng(6).normal(size=(r, 3))))
    cfg = render.RenderConfig(0.05, 200.0, render.RenderMode.RGB, n, k, density_shift=0.0)

    def gradients(rows):
        rays = cameras.Rays3D(o[rows], d[rows],
                              torch.zeros(o[rows].shape[0], dtype=torch.int32, device="cuda"))
        out = render.render_rays(mlp_module(shape), lp, dev(np.array([[-1.5] * 3, [1.5] * 3])),
                                 rays, 3, cfg)
        return torch.autograd.grad((out * up[rows]).sum(), leaves)

    whole = gradients(slice(0, r))
    sums = [torch.zeros_like(t, dtype=torch.float64) for t in leaves]
    for at in range(0, r, part):
        for s, t in zip(sums, gradients(slice(at, min(r, at + part)))):
            s += t.double()
    for name, t, s in zip(("density plane", "density line", "appearance plane",
                           "appearance line"), whole, sums):
        e = report(name, t.cpu().numpy(), s.cpu().numpy())
        assert e.max() <= 2e-4 * float(s.abs().max()) + 1e-7, name
