"""The MLP backward of the fused training step at row counts around its tiles
(32 rows in FP32, 64 in BF16; kept activations in groups of 32 rows): one row,
a row short of and past a tile, and a tile that spans rays and cameras.

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


@pytest.mark.parametrize("film", [False, True])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rays,samples", [(1, 1), (1, 31), (4, 8), (3, 11), (1, 63), (2, 32),
                                          (5, 13), (7, 37)])
def test_train_step_gradient_at_tile_edges(rays, samples, precision, film):
    log(f"case: {rays} rays x {samples} samples, {precision}, FiLM {film}")
    from tensorf_amd import cameras, render, training
    g, ncam = 12, 3
    shape = orc.MlpShape(num_cameras=ncam if film else None)
    cfg = training.TensorfConfig(
        minibatch_size=rays, n_iters=100, initial_aabb_min=(-1.5,) * 3,
        initial_aabb_max=(1.5,) * 3, appearance_feat_dim=48, density_feat_dim=16,
        feature_n_freqs=2, viewdir_n_freqs=2, grid_dim_init=g, grid_dim_final=g, upsamp_iters=(),
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
