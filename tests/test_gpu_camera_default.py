"""The C interface takes null camera indices for camera 0 where the MLP has a
camera embedding: every render and training entry point gives what zero indices
give, for the shapes with compile-time dims (48 channels with 2 frequencies, 24
with 6) and another one, on tiles that span rays and tiles within one. Outputs
bit for bit; gradients to 1e-5 of the largest (float adds in any order)."""
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import log, report

pytestmark = pytest.mark.gpu

SHAPES = [(48, 2), (24, 6), (20, 3)]


def _state(channels, freqs, precision, rays, samples, proposal=None):
    from tensorf_amd import training
    cfg = training.TensorfConfig(
        minibatch_size=rays, n_iters=100, initial_aabb_min=(-1.5,) * 3,
        initial_aabb_max=(1.5,) * 3, appearance_feat_dim=channels, density_feat_dim=16,
        feature_n_freqs=freqs, viewdir_n_freqs=freqs, grid_dim_init=12, grid_dim_final=12,
        upsamp_iters=(), density_samples_per_ray=samples, appearance_samples_per_ray=samples,
        camera_embeddings=True, mlp_precision=precision, density_shift=0.0, proposal=proposal)
    return training.TrainState.initialize(cfg, 12, prng_key=3, num_cameras=3)


def _rays(rays):
    from tensorf_amd import cameras
    o, d = orc.make_rays(rays, seed=8, radius=4.0, target_half=0.5)
    return cameras.Rays3D(torch.tensor(o, dtype=torch.float32, device="cuda"),
                          torch.tensor(d, dtype=torch.float32, device="cuda"),
                          torch.zeros(rays, dtype=torch.int32, device="cuda"))


def _with_and_without(monkeypatch, run):
    """run() with zero camera indices, then with a null pointer for them."""
    from tensorf_amd import render
    want = run()
    init = render._RenderEnv.__init__

    def no_cameras(self, *args, **kwargs):
        init(self, *args, **kwargs)
        self.cams = None

    monkeypatch.setattr(render._RenderEnv, "__init__", no_cameras)
    return want, run()


def _same(name, got, want):
    e = report(name, got.cpu().numpy(), want.cpu().numpy())
    assert e.max() <= 1e-5 * float(want.abs().max()), name


@pytest.mark.parametrize("channels,freqs", SHAPES)
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rays,samples", [(9, 7), (3, 70)])
def test_render_and_its_gradient(monkeypatch, rays, samples, precision, channels, freqs):
    log(f"case: render, {rays} rays x {samples}, {channels} channels, {precision}")
    from tensorf_amd import render
    st = _state(channels, freqs, precision, rays, samples)
    batch, lp = _rays(rays), st.learnable_params
    env_leaves = render._RenderEnv(st.appearance_mlp, lp, st.aabb, batch, 5, st.render_config(),
                                   alloc_workspace=False).leaves()
    leaves = [t.requires_grad_(True) for t in env_leaves]
    up = torch.randn(rays, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(1))

    def run():
        args = (st.appearance_mlp, lp, st.aabb, batch, 5, st.render_config())
        with torch.no_grad():
            only = render.render_rays(*args)
        out = render.render_rays(*args)
        return [only, out.detach(), *torch.autograd.grad(out, leaves, up)]

    want, got = _with_and_without(monkeypatch, run)
    assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])
    for i, (w, g) in enumerate(zip(want[2:], got[2:])):
        _same(f"gradient {i}", g, w)
    assert float(want[-1][0].abs().max()) > 0 and float(want[-1][1:].abs().max()) == 0


@pytest.mark.parametrize("channels,freqs", SHAPES)
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("with_proposal", [False, True])
def test_training_step(monkeypatch, with_proposal, precision, channels, freqs):
    log(f"case: training step, {channels} channels, {precision}, proposal {with_proposal}")
    from tensorf_amd import cameras, proposal
    rays, samples = 11, 32
    pc = proposal.ProposalConfig(samples_round0=16, samples_round1=16, samples_out=samples,
                                 grid_dim=12) if with_proposal else None
    batch = cameras.RenderedRays(torch.full((rays, 3), 0.25, device="cuda"), _rays(rays))

    def run():
        st = _state(channels, freqs, precision, rays, samples, pc)
        _, logs = st.training_step(batch)
        return logs["mse"].clone(), st.flat.exp_avg.clone()

    (mse, avg), (mse_null, avg_null) = _with_and_without(monkeypatch, run)
    assert float((mse - mse_null).abs()) <= 1e-6 * float(mse)
    _same("first moment", avg_null, avg)


@pytest.mark.parametrize("channels,freqs", SHAPES)
def test_forward_without_allocation(monkeypatch, channels, freqs):
    log(f"case: forward without allocation, {channels} channels")
    import ctypes

    from tensorf_amd import _lib, render
    rays = 9
    st = _state(channels, freqs, "fp32", rays, 7)

    def run():
        env = render._RenderEnv(st.appearance_mlp, st.learnable_params, st.aabb, _rays(rays), 5,
                                st.render_config(), alloc_workspace=False)
        out = torch.zeros(rays, 3, device="cuda")
        _lib.call("tfh_render_fwd_noalloc", ctypes.byref(env.dvm), ctypes.byref(env.avm),
                  env._mlp_ref(), ctypes.byref(env.cfg), _lib.ptr(env.aabb), _lib.ptr(env.o),
                  _lib.ptr(env.d), _lib.ptr(env.cams), rays, _lib.ptr(env.jitter),
                  _lib.ptr(env.base_ts), _lib.ptr(env.base_steps), _lib.ptr(env.gumbel),
                  _lib.ptr(out), _lib.stream())
        return out

    want, got = _with_and_without(monkeypatch, run)
    assert torch.equal(want, got)
