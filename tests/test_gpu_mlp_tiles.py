"""The MLP backward of the fused training step at row counts around its tiles
(32 rows in FP32, 64 in BF16; kept activations in groups of 32 rows): one row,
a row short of and past a tile, and a tile that spans rays and cameras; for both
shapes with compile-time dims (48 channels with 2 frequencies, 24 with 6).

The step's gradient is read back from Adam's first moment (0.1 g after the
first step) and compared with the float64 oracle's: FP32 within 2e-4 of the
largest gradient of the group (summation order of at most a few hundred rows,
as in the other gradient tests); BF16 against the oracle with the same operand
rounding, within 2e-2 of the largest for all but 1e-3 of the elements and 1e-2
relative L2 (isolated rounding ties)."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, report

pytestmark = pytest.mark.gpu

NAMES = ["density_matrix", "density_vector", "appearance_matrix", "appearance_vector",
         "w0", "w1", "b1", "w2", "b2", "w3", "b3", "embed"]


def _reference_layout(flat, buf):
    out = {}
    for i, name in enumerate(NAMES[:len(flat.names)]):
        t = flat.view(buf, i)
        if name.endswith("matrix"):
            t = t.permute(0, 3, 1, 2)
        elif name.endswith("vector"):
            t = t.permute(0, 2, 1)
        out[name] = t.cpu().numpy().astype(np.float64)
    return out


@pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])
@pytest.mark.parametrize("film", [False, True])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rays,samples", [(1, 1), (1, 31), (4, 8), (3, 11), (1, 63), (2, 32),
                                          (5, 13), (7, 37)])
def test_train_step_gradient_at_tile_edges(rays, samples, precision, film, channels, freqs):
    log(f"case: {rays} rays x {samples} samples, {precision}, FiLM {film}, {channels} channels")
    from tensorf_amd import cameras, render, training
    g, ncam = 12, 3
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs,
                         num_cameras=ncam if film else None)
    cfg = training.TensorfConfig(
        minibatch_size=rays, n_iters=100, initial_aabb_min=(-1.5,) * 3,
        initial_aabb_max=(1.5,) * 3, appearance_feat_dim=channels, density_feat_dim=16,
        feature_n_freqs=freqs, viewdir_n_freqs=freqs, grid_dim_init=g, grid_dim_final=g, upsamp_iters=(),
        density_samples_per_ray=samples, appearance_samples_per_ray=samples,
        camera_embeddings=film, mlp_precision=precision, density_shift=0.0)
    st = training.TrainState.initialize(cfg, g, prng_key=3, num_cameras=ncam)
    gen = torch.Generator().manual_seed(1)
    for i in (6, 8, 10):  # biases away from zero
        v = st.flat.view(st.flat.params, i)
        v.copy_(0.1 * torch.randn(v.shape, generator=gen))
    p = _reference_layout(st.flat, st.flat.params)
    o, d = orc.make_rays(rays, seed=8, radius=4.0, target_half=0.5)
    o, d = f32(o), f32(d)
    cams = np.arange(rays) % ncam
    colors = f32(np.random.default_rng(8).uniform(size=(rays, 3)))
    batch = cameras.RenderedRays(dev(colors), cameras.Rays3D(dev(o), dev(d),
                                                             dev(cams, torch.int32)))
    seed = render._seed(st.prng_key, 0)
    jit = render.uniform(render._seed(seed, 1), samples).cpu().numpy().astype(np.float64)
    st.training_step(batch)
    got = {k: 10.0 * v for k, v in _reference_layout(st.flat, st.flat.exp_avg).items()}
    ocfg = orc.RenderConfig(0.05, 200.0, orc.RGB, samples, samples, density_shift=0.0)
    out, cache = orc.render_rays(p, np.array([[-1.5] * 3, [1.5] * 3]), o, d, cams, ocfg, shape,
                                 jit, mlp_operand_round=orc.bf16_round if precision == "bf16"
                                 else None)
    want = orc.render_rays_backward(p, cache, 2.0 * (out - colors) / out.size, ocfg, shape)
    for name, val in got.items():
        e = report(f"grad {name}", val, want[name])
        top = np.abs(want[name]).max()
        if precision == "fp32":
            assert e.max() <= 2e-4 * top + 1e-9, name
        else:
            assert (e > 2e-2 * top + 1e-9).mean() <= 1e-3, name
            assert np.linalg.norm(e) <= 1e-2 * np.linalg.norm(want[name]) + 1e-9, name


@pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])
@pytest.mark.parametrize("ncam", [None, 3])
@pytest.mark.parametrize("rows", [1, 33, 131072 + 33])
def test_mlp_backward_across_chunks(rows, ncam, channels, freqs):
    """FeatureMlp.apply's backward runs the forward and the backward in chunks
    of 131,072 rows: a batch one tile and a row past a chunk gives each row's
    feature gradient as a one-row batch would (torch float64, 1e-4 of the
    largest, checked on the rows around the chunk's end), and the weight
    gradients sum over both chunks (the bias gradient b3 of all rows)."""
    log(f"case: {rows} rows, cameras {ncam}, {channels} channels")
    from tests.gpu_common import mlp_module, oracle_params, to_device_params
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs,
                         num_cameras=ncam)
    p = oracle_params(4, 16, channels, shape, seed=3, bias_std=0.1)
    _, _, mp = to_device_params(p, shape)
    mlp = mlp_module(shape)
    gen = torch.Generator("cuda").manual_seed(2)
    f = (0.3 * torch.randn(rows, 3 * channels, device="cuda", generator=gen)).requires_grad_(True)
    d = torch.randn(rows, 3, device="cuda", generator=gen)
    cams = torch.randint(0, ncam or 1, (rows,), device="cuda", generator=gen).to(torch.int32)
    up = torch.randn(rows, 3, device="cuda", generator=gen)
    leaves = [t.requires_grad_(True) for t in mlp.flat_leaves(mp)]
    rgb = mlp.apply(mp, f, d, cams)
    grads = torch.autograd.grad(rgb, [f, *leaves], up)
    at = np.unique(np.clip(np.r_[0:4, rows - 40:rows], 0, rows - 1))
    want, cache = orc.feature_mlp_forward(p, f.detach()[at].cpu().numpy(), d[at].cpu().numpy(),
                                          cams[at].cpu().numpy(), shape)
    _, gf = orc.feature_mlp_backward(p, cache, up[at].cpu().numpy(), shape)
    e = report("grad features", grads[0][at].cpu().numpy(), gf)
    assert e.max() <= 1e-4 * np.abs(gf).max() + 1e-6
    s = rgb.detach().double()
    b3 = (up.double() * s * (1 - s)).sum(0).cpu().numpy()
    assert report("grad b3", grads[7].cpu().numpy(), b3).max() <= 1e-4 * np.abs(b3).max() + 1e-4
