"""A render without a backward to follow gives the same bits as one that keeps the
backward's residuals: shapes whose gather is inside the MLP kernel and not, all
samples shaded or the top k, and the distance modes."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, mlp_module, oracle_params, to_device_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["RGB", "DIST_MEDIAN", "DIST_MEAN"])
@pytest.mark.parametrize("ca,precision", [(48, "fp32"), (48, "bf16"), (8, "fp32")])
@pytest.mark.parametrize("n,k", [(70, 70), (70, 9)])
def test_same_bits(n, k, ca, precision, mode):
    log(f"case: {mode}, {n} samples, {k} shaded, {ca} channels, {precision}")
    from tensorf_amd import cameras, render
    r, shape = 41, orc.MlpShape(feat_dim=3 * ca)
    p = oracle_params(12, 8, ca, shape, seed=5, std=0.5, bias_std=0.1)
    den, app, mp = to_device_params(p, shape)
    lp = render.LearnableParams(mp, app, den, False)
    o, d = orc.make_rays(r, seed=4, radius=3.0, target_half=1.2)
    rays = cameras.Rays3D(dev(f32(o)), dev(f32(d)),
                          torch.zeros(r, dtype=torch.int32, device="cuda"))
    box = dev(np.array([[-1.5] * 3, [1.5] * 3]))
    cfg = render.RenderConfig(0.05, 200.0, render.RenderMode[mode], n, k, density_shift=0.0)
    env = render._RenderEnv(mlp_module(shape, precision), lp, box, rays, 3, cfg)
    with torch.no_grad():
        kept = env.forward()
        env.ws.fill_(255)  # nothing that is read may be left from before
        only = env.forward(keep=False)
    assert torch.equal(kept, only) or (torch.isnan(kept) == torch.isnan(only)).all()
    assert torch.equal(torch.nan_to_num(kept), torch.nan_to_num(only))
