"""The MLP backward of callers that kept no activations goes in chunks of 131,072
rows (of whole rays): every gradient of a batch past a chunk, a tile and a row is
the float64 sum of the gradients of parts that are smaller than a chunk, for the MLP
by itself and inside a render. Parts and batch form the same products per row, so
they differ by the order of FP32 sums (2e-4 of the largest of a gradient, as in the
other tests; a chunk lost or counted twice shows at 1e-2)."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, mlp_module, oracle_params, report, to_device_params

pytestmark = pytest.mark.gpu

CHUNK = 131072
KEYS = ["w0", "w1", "b1", "w2", "b2", "w3", "b3", "embed"]


def _compare(names, whole, parts):
    for name, w, s in zip(names, whole, parts):
        e = report(name, w.cpu().numpy(), s.cpu().numpy())
        assert e.max() <= 2e-4 * float(s.abs().max()), name


@pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])
@pytest.mark.parametrize("ncam", [None, 3])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rows", [CHUNK + 33, 2 * CHUNK + 1])
def test_mlp(rows, precision, ncam, channels, freqs):
    log(f"case: {rows} rows, cameras {ncam}, {channels} channels, {precision}")
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs,
                         num_cameras=ncam)
    p = oracle_params(4, 16, channels, shape, seed=3, bias_std=0.1)
    _, _, mp = to_device_params(p, shape)
    mlp = mlp_module(shape, precision)
    gen = torch.Generator("cuda").manual_seed(2)
    f = 0.3 * torch.randn(rows, 3 * channels, device="cuda", generator=gen)
    d = torch.randn(rows, 3, device="cuda", generator=gen)
    cams = torch.randint(0, ncam or 1, (rows,), device="cuda", generator=gen).to(torch.int32)
    up = torch.randn(rows, 3, device="cuda", generator=gen)
    leaves = [t.requires_grad_(True) for t in mlp.flat_leaves(mp)]

    def gradients(a, b):
        x = f[a:b].clone().requires_grad_(True)
        return torch.autograd.grad(mlp.apply(mp, x, d[a:b], cams[a:b]), [x, *leaves], up[a:b])

    whole = gradients(0, rows)
    sums = [torch.zeros_like(t, dtype=torch.float64) for t in leaves]
    features = []
    for at in range(0, rows, 50000):
        part = gradients(at, min(at + 50000, rows))
        features.append(part[0].double())
        for s, g in zip(sums, part[1:]):
            s += g.double()
    _compare(["features", *KEYS], whole, [torch.cat(features), *sums])


@pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rays,samples", [(1050, 130)])
def test_render(rays, samples, precision, channels, freqs):
    """A chunk ends within the batch and holds whole rays (1008 of 130 samples)."""
    log(f"case: {rays} rays x {samples}, {channels} channels, {precision}")
    from tensorf_amd import cameras, render
    assert rays * samples > CHUNK > (CHUNK // samples) * samples
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs,
                         num_cameras=3)
    p = oracle_params(16, 8, channels, shape, seed=5, std=0.3, bias_std=0.1)
    den, app, mp = to_device_params(p, shape)
    lp = render.LearnableParams(mp, app, den, False)
    o, d = orc.make_rays(rays, seed=4, radius=3.0, target_half=0.6)
    batch = cameras.Rays3D(dev(f32(o)), dev(f32(d)), dev(np.arange(rays) % 3, torch.int32))
    box = dev(np.array([[-1.5] * 3, [1.5] * 3]))
    cfg = render.RenderConfig(0.05, 200.0, render.RenderMode.RGB, samples, samples,
                              density_shift=0.0)
    mlp = mlp_module(shape, precision)
    leaves = [t.requires_grad_(True) for t in render._leaves(lp)]
    up = torch.randn(rays, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(1))

    def gradients(a, b):
        out = render.render_rays(mlp, lp, box, batch.slice(a, b), 3, cfg)
        return torch.autograd.grad(out, leaves, up[a:b])

    whole = gradients(0, rays)
    sums = [torch.zeros_like(t, dtype=torch.float64) for t in leaves]
    for at in range(0, rays, 350):
        for s, g in zip(sums, gradients(at, min(at + 350, rays))):
            s += g.double()
    _compare(["density plane", "density line", "appearance plane", "appearance line", *KEYS],
             whole, sums)
