"""The density pass at sample counts around its chunks of 64 and at the channel
counts that choose its lanes per sample (2, 4, 8, 16 with 16-byte taps; 16 with
4-byte ones), in every mode it serves. Tolerances as in the other render tests:
1e-5 relative of the oracle; a median may move where 1 - E is within 1e-5 of
0.5, a top-k choice where two weights tie within FP32."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, mlp_module, oracle_params, report, to_device_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["rgb", "median", "mean"])
@pytest.mark.parametrize("channels", [4, 8, 12, 20, 36, 3, 18])
@pytest.mark.parametrize("n,k", [(1, 1), (63, 20), (64, 64), (65, 65), (130, 9)])
def test_chunk_edges(n, k, channels, mode):
    log(f"case: {mode}, {n} samples, {k} shaded, {channels} channels")
    from tensorf_amd import cameras, render
    g, r = 12, 37
    shape = orc.MlpShape(feat_dim=24)
    p = oracle_params(g, channels, 8, shape, seed=5, std=0.5, bias_std=0.1)
    p["density_matrix"] = p["density_matrix"] * 4.0  # medians inside the box
    den, app, mp = to_device_params(p, shape)
    lp = render.LearnableParams(mp, app, den, False)
    o, d = orc.make_rays(r, seed=4, radius=3.0, target_half=1.2)
    o, d = f32(o), f32(d)
    box = np.array([[-1.5] * 3, [1.5] * 3])
    rays = cameras.Rays3D(dev(o), dev(d), torch.zeros(r, dtype=torch.int32, device="cuda"))
    gpu_mode, oracle_mode = {"rgb": (render.RenderMode.RGB, orc.RGB),
                             "median": (render.RenderMode.DIST_MEDIAN, orc.DIST_MEDIAN),
                             "mean": (render.RenderMode.DIST_MEAN, orc.DIST_MEAN)}[mode]
    cfg = render.RenderConfig(0.05, 200.0, gpu_mode, n, k, density_shift=0.0)
    with torch.no_grad():
        out = render.render_rays(mlp_module(shape), lp, dev(box), rays, 3, cfg).cpu().numpy()
    jit = render.uniform(render._seed(3, 1), n).cpu().numpy().astype(np.float64)
    ocfg = orc.RenderConfig(0.05, 200.0, oracle_mode, n, k, density_shift=0.0)
    want, cache = orc.render_rays(p, box, o, d, np.zeros(r), ocfg, shape, jit)
    skip = np.zeros(r, dtype=bool)
    if mode == "median":
        skip = np.any(np.abs(0.5 - cache["p_exits"]) < 1e-5, axis=1)
        assert np.array_equal(np.isinf(out)[~skip], np.isinf(want)[~skip])
        skip |= np.isinf(want)
    elif mode == "rgb" and k < n:
        srt = np.sort(cache["w"], axis=1)[:, ::-1]
        skip = np.abs(srt[:, k - 1] - srt[:, k]) < 1e-5 * np.maximum(srt[:, k - 1], 1e-30)
    assert skip.mean() < 1.0 or mode == "median"
    report(mode, out[~skip], want[~skip])
    np.testing.assert_allclose(out[~skip], want[~skip], rtol=1e-5, atol=2e-6)
