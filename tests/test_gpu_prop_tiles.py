"""The proposal MLP around its tiles: 32 rows per wave (16 in the backward) and 8
waves per workgroup, 6 first-layer products up to 24 features and 8 past them, and the field gather
inside it (8 channels) or before it (other channel counts). Tolerances are those
of the other proposal tests: FP32 sums of up to 64 products, 2e-5 of the largest
output; weights at the sampler's own intervals 1e-4."""
import numpy as np
import pytest

from oracle import proposal_oracle as po
from tests.gpu_common import dev, f32, log, report
from tests.test_gpu_proposal import _device_field, _prop_params, _rays, _sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels", [1, 5, 8, 9, 10])
@pytest.mark.parametrize("rows", [1, 15, 17, 32, 33, 255, 257, 20000])
def test_forward_at_tile_edges(rows, channels):
    log(f"case: proposal mlp, {rows} rows, {3 * channels} features")
    from tensorf_amd import proposal
    pp = _prop_params(c=channels)
    feats = f32(np.random.default_rng(rows).normal(0, 0.5, (rows, 3 * channels)))
    z, sig = proposal.mlp_forward(_device_field(pp).mlp, dev(feats))
    zr, sr, _ = po.prop_mlp_forward(pp, feats)
    assert report("z", z.cpu().numpy(), zr).max() <= 2e-5 * max(1.0, np.abs(zr).max())
    assert report("sigma", sig.cpu().numpy(), sr).max() <= 2e-5 * max(1.0, np.abs(sr).max())


@pytest.mark.parametrize("channels", [1, 5, 8, 9, 10])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 127, 129, 5000])
def test_backward_at_tile_edges(rows, channels):
    log(f"case: proposal mlp backward, {rows} rows, {3 * channels} features")
    from tensorf_amd import proposal
    pp = _prop_params(c=channels)
    rng = np.random.default_rng(rows)
    feats = f32(rng.normal(0, 0.5, (rows, 3 * channels)))
    dz = f32(rng.normal(size=rows))
    grads, gf = proposal.mlp_backward(_device_field(pp).mlp, dev(feats), dev(dz))
    _, _, cache = po.prop_mlp_forward(pp, feats)
    gr, gfr = po.prop_mlp_backward(pp, cache, dz)
    for k in proposal.MLP_KEYS:
        e = report(f"d{k}", grads[k].cpu().numpy(), gr["p" + k])
        assert e.max() <= 1e-4 * np.abs(gr["p" + k]).max() + 1e-6
    e = report("dfeat", gf.cpu().numpy(), gfr)
    assert e.max() <= 1e-4 * np.abs(gfr).max()


@pytest.mark.parametrize("rays", [1, 3, 37])
@pytest.mark.parametrize("channels", [4, 8, 9])
def test_sampler_gathers_the_field(channels, rays):
    log(f"case: {channels} channels, {rays} rays")
    cfg = po.ProposalConfig(samples_round0=37, samples_round1=11, samples_out=9)
    pp = _prop_params(c=channels)
    o, d = _rays(rays, 5)
    jit = f32(np.random.default_rng(5).uniform(size=(rays, 48)))
    s, field, box, keep = _sample(pp, cfg, o, d, jit, False, None, None, 1.0)
    edges = [s.round(k)[0].cpu().numpy().astype(np.float64) for k in range(2)]
    _, rounds = po.proposal_rounds(pp, cfg, box, o, d, jit, None, None, edges)
    for k in range(2):
        e = report(f"round {k} weights", s.round(k)[1].cpu().numpy(), rounds[k]["w"])
        assert e.max() <= 1e-4
