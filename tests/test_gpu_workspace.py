"""What the workspaces hold. A training step that keeps its activations reserves no
second place for them, a render without a backward nothing of the backward's, the
BF16 MLP's activations take 16 bits a value (sizes, on the CPU); and a render in a
workspace of exactly its size gives the bits of one that a backward can follow, and
leaves the memory behind it alone (on the GPU)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, mlp_module, oracle_params, to_device_params

LINES = (8 << 20) + (4 << 20)  # copies of the factor-line gradients
SLACK = 1 << 21                # weight tables, rounding up


def _sizes(rays, n, k, precision=0, mode=0, channels=48, freqs=2, cams=0):
    from tensorf_amd import _lib
    cfg = _lib.RenderConfig(0.05, 200.0, mode, n, k, 0, precision, 0, 0.0)
    mlp = _lib.Mlp(*([256] * 7), 256 if cams else None, 3 * channels, 27, 128, freqs, freqs, cams)

    def size(name):
        return getattr(_lib.lib, name)(ctypes.byref(cfg), ctypes.byref(mlp), channels, rays)

    return [size(f"tfh_{name}_workspace_size") for name in ("render", "render_only", "train_step")]


@pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])
@pytest.mark.parametrize("rays,n,k", [(64, 32, 32), (4096, 221, 33), (4096, 512, 512),
                                      (8192, 512, 64)])
def test_sizes(rays, n, k, channels, freqs):
    rows, samples, f = rays * k, rays * n, 3 * channels
    chunk = min(rows, 131072)  # rows whose activations a backward forms at a time
    fp32 = _sizes(rays, n, k, 0, channels=channels, freqs=freqs)
    bf16 = _sizes(rays, n, k, 1, channels=channels, freqs=freqs)
    # per sample: point, density, step, weight, transmittance, gradient, sort; per
    # row: features and their gradient, colour and its gradient; per workgroup the
    # weight gradients (68,891 values of the wide shape)
    backward = samples * (12 + 4 * 4 + 4 + 30) + rows * (8 * f + 24 + 4) + 256 * 4 * 69000
    assert fp32[0] <= backward + chunk * (1024 + 12) + SLACK + 64 * rays
    assert fp32[1] <= samples * 28 + rows * (4 * f + 12 + 4) + 16 * rays + SLACK
    for sizes, kept in ((fp32, 1024), (bf16, 512)):
        act, again = rows * kept, chunk * (kept + 12)
        assert sizes[2] - sizes[0] <= max(act - again, 0) + LINES + (1 << 16)


@pytest.mark.parametrize("mode", [1, 2, 3])
def test_distances_reserve_no_shading(mode):
    only = _sizes(4096, 512, 512, 0, mode)[1]
    assert 0 < only <= 4096 * (512 * 28 + 16) + (1 << 16)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["RGB", "DIST_MEDIAN", "DIST_MEAN"])
@pytest.mark.parametrize("ca,freqs,precision", [(48, 2, "fp32"), (48, 2, "bf16"), (24, 6, "fp32"),
                                                (20, 3, "bf16")])
@pytest.mark.parametrize("r,n,k", [(41, 70, 70), (41, 70, 9), (1, 1, 1)])
def test_render_stays_in_its_workspace(r, n, k, ca, freqs, precision, mode):
    log(f"case: {mode}, {r} rays, {n} samples, {k} shaded, {ca} channels, {precision}")
    from tensorf_amd import cameras, render
    shape = orc.MlpShape(feat_dim=3 * ca, feature_n_freqs=freqs, viewdir_n_freqs=freqs)
    p = oracle_params(12, 8, ca, shape, seed=5, std=0.5, bias_std=0.1)
    den, app, mp = to_device_params(p, shape)
    lp = render.LearnableParams(mp, app, den, False)
    o, d = orc.make_rays(r, seed=4, radius=3.0, target_half=1.2)
    rays = cameras.Rays3D(dev(f32(o)), dev(f32(d)),
                          torch.zeros(r, dtype=torch.int32, device="cuda"))
    box = dev(np.array([[-1.5] * 3, [1.5] * 3]))
    cfg = render.RenderConfig(0.05, 200.0, render.RenderMode[mode], n, k, density_shift=0.0)
    mlp = mlp_module(shape, precision)
    want = render._RenderEnv(mlp, lp, box, rays, 3, cfg).forward()
    env = render._RenderEnv(mlp, lp, box, rays, 3, cfg, keep=False)
    size = env.ws.numel()
    both = torch.full((size + 65536,), 255, dtype=torch.uint8, device="cuda")
    env.ws = both[:size]
    got = env.forward()
    assert torch.equal(torch.isnan(want), torch.isnan(got))
    assert torch.equal(torch.nan_to_num(want), torch.nan_to_num(got))
    assert bool((both[size:] == 255).all())
