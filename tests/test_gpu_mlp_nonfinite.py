"""The FP32 MLP backward forms most of its products from BF16 planes of its
operands, which cannot hold infinities or values above BF16's largest: such
batches are done again with FP32 products. Gradients of a batch with an infinite
upstream gradient in one row have infinities of the same sign and NaN at the
same places as the formulas in float64 give them, and the other values; a
feature near FLT_MAX that its weights ignore leaves every gradient finite.

Finite values within 2e-4 of the largest of their gradient (the tolerance of the
other gradient tests: summation order). No pre-activation of the rows with an
infinity is within 1e-5 of a ReLU's edge; what the other rows of a batch add is the
library's own gradient without that row's (at an edge float32 and float64 may
differ in whether a unit passes its gradient)."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, mlp_module, oracle_params, to_device_params

pytestmark = pytest.mark.gpu

KEYS = ["w0", "w1", "b1", "w2", "b2", "w3", "b3", "embed"]


def _mul(a, b):
    """a @ b with every product formed (0 * inf is NaN)."""
    return np.einsum("ij,jk->ik", a, b, optimize=False)


def _backward(p, c, grad_rgb, shape):
    """The oracle's backward (networks.py:46-121) with selections for the ReLUs,
    which pass no gradient, infinite or not, where they are off."""
    with np.errstate(invalid="ignore", over="ignore"):
        dz3 = grad_rgb * c["rgb"] * (1.0 - c["rgb"])
        g = {"w3": _mul(c["h2f"].T, dz3), "b3": dz3.sum(0)}
        dh2 = _mul(dz3, p["w3"].T)
        if shape.num_cameras is not None:
            half = shape.units // 2
            rows = np.concatenate([dh2[:, half:] * c["h2"][:, half:], dh2[:, half:]], -1)
            g["embed"] = np.zeros_like(p["embed"])
            np.add.at(g["embed"], c["cams"], rows)
            dh2[:, half:] *= c["emb"][:, :half]
        dz2 = np.where(c["z2"] > 0, dh2, 0.0)
        g["w2"], g["b2"] = _mul(c["h1"].T, dz2), dz2.sum(0)
        dz1 = np.where(c["z1"] > 0, _mul(dz2, p["w2"].T), 0.0)
        g["w1"], g["b1"] = _mul(c["x"].T, dz1), dz1.sum(0)
        dx = _mul(dz1, p["w1"].T)
        sq, nf, h0 = shape.squash_dim, shape.feature_n_freqs, c["h0"]
        dh0 = dx[:, :sq].copy()
        fe = dx[:, sq + 3:sq + 3 + 2 * nf * sq].reshape(-1, sq, 2 * nf)
        for q in range(nf):
            s = 2.0 ** q
            dh0 += fe[:, :, q] * s * np.cos(s * h0) - fe[:, :, nf + q] * s * np.sin(s * h0)
        g["w0"] = _mul(c["f"].T, dh0)
        return g, _mul(dh0, p["w0"].T)


def _check(name, got, want):
    got = np.asarray(got, np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)), name
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf]), name
    ok = np.isfinite(want)
    top = np.abs(want[ok]).max() if ok.any() else 0.0
    err = np.abs(got[ok] - want[ok]).max() if ok.any() else 0.0
    log(f"  {name}: {int(inf.sum())} infinite, {int(np.isnan(want).sum())} NaN, "
        f"{int(ok.sum())} finite, max|err|={err:.3e} of {top:.3e}")
    assert err <= 2e-4 * top + 1e-9, name


def _clear(c):
    """Rows with no pre-activation at a ReLU's edge."""
    return np.minimum(np.abs(c["z1"]).min(1), np.abs(c["z2"]).min(1)) > 1e-5


def _mlp_gradients(p, shape, f, d, cams, up):
    _, _, mp = to_device_params(p, shape)
    mlp = mlp_module(shape)
    leaves = [t.requires_grad_(True) for t in mlp.flat_leaves(mp)]
    fd = dev(f).requires_grad_(True)
    rgb = mlp.apply(mp, fd, dev(d), dev(cams, torch.int32))
    grads = torch.autograd.grad(rgb, [fd, *leaves], dev(up))
    return [t.cpu().numpy() for t in grads]


def _rows(rows, shape, seed):
    rng = np.random.default_rng(seed)
    f = f32(rng.normal(0, 0.3, (rows, shape.feat_dim)))
    d = f32(rng.normal(size=(rows, 3)))
    cams = rng.integers(0, shape.num_cameras or 1, rows)
    return f, d, cams, f32(rng.normal(size=(rows, 3)))


SHAPES = pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])


@SHAPES
@pytest.mark.parametrize("ncam", [None, 3])
@pytest.mark.parametrize("rows,at,value", [(1, 0, np.inf), (70, 41, -np.inf), (70, 69, np.inf),
                                           (9001, 8999, -np.inf)])
def test_infinite_upstream_gradient(rows, at, value, ncam, channels, freqs):
    log(f"case: {value} in row {at} of {rows}, cameras {ncam}, {channels} channels")
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs,
                         num_cameras=ncam)
    p = oracle_params(4, 16, channels, shape, seed=3, bias_std=0.1)
    f, d, cams, up = _rows(rows, shape, 5)
    up[at, 1] = value
    got = _mlp_gradients(p, shape, f, d, cams, up)
    # the row by itself holds every value that is not finite
    _, one = orc.feature_mlp_forward(p, f[at:at + 1], d[at:at + 1], cams[at:at + 1], shape)
    assert _clear(one).all()
    want, gf = _backward(p, one, up[at:at + 1], shape)
    _check("features of the row", got[0][at:at + 1], gf)
    finite = up.copy()
    finite[at] = 0.0
    other = _mlp_gradients(p, shape, f, d, cams, finite)
    rest = np.delete(np.arange(rows), at)
    if rows > 1:
        _check("features of the others", got[0][rest], other[0][rest])
    for key, val, add in zip(KEYS, got[1:], other[1:]):
        with np.errstate(invalid="ignore"):
            _check(key, val, want[key] + add)


@SHAPES
@pytest.mark.parametrize("ncam", [None, 3])
def test_feature_that_bf16_cannot_hold(ncam, channels, freqs):
    """3.4e38 rounds to infinity in BF16; a weight row of zeros keeps it out of
    the forward, and its weight gradient is 3.4e38 dL/dh0."""
    log(f"case: a feature of 3.4e38, cameras {ncam}, {channels} channels")
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs,
                         num_cameras=ncam)
    p = oracle_params(4, 16, channels, shape, seed=3, bias_std=0.1)
    p["w0"][5] = 0.0
    f, d, cams, up = _rows(70, shape, 5)
    f[33, 5] = float(np.float32(3.4e38))
    up = f32(1e-3 * up)
    got = _mlp_gradients(p, shape, f, d, cams, up)
    _, c = orc.feature_mlp_forward(p, f, d, cams, shape)
    want, gf = orc.feature_mlp_backward(p, c, up, shape)
    assert np.abs(want["w0"]).max() < 3e38
    _check("features", got[0], gf)
    for key, val in zip(KEYS, got[1:]):
        if key == "w0":
            _check("w0, the feature's row", val[5:6], want[key][5:6])
            _check("w0, the others", np.delete(val, 5, 0), np.delete(want[key], 5, 0))
        else:
            _check(key, val, want[key])


@SHAPES
def test_weight_that_bf16_cannot_hold(channels, freqs):
    """A weight of 3.4e38 that only meets features of zero: dL/df of that feature
    is 3.4e38 dL/dh0, the rest is as without it."""
    log(f"case: a weight of 3.4e38, {channels} channels")
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs)
    p = oracle_params(4, 16, channels, shape, seed=3, bias_std=0.1)
    p["w0"][7, 3] = float(np.float32(3.4e38))
    f, d, cams, up = _rows(70, shape, 5)
    f[:, 7] = 0.0
    up = f32(1e-3 * up)
    got = _mlp_gradients(p, shape, f, d, cams, up)
    _, c = orc.feature_mlp_forward(p, f, d, cams, shape)
    want, gf = orc.feature_mlp_backward(p, c, up, shape)
    assert np.abs(gf).max() < 3e38
    _check("dL/df of the feature", got[0][:, 7:8], gf[:, 7:8])
    _check("dL/df of the others", np.delete(got[0], 7, 1), np.delete(gf, 7, 1))
    for key, val in zip(KEYS, got[1:]):
        _check(key, val, want[key])


@SHAPES
@pytest.mark.parametrize("film", [False, True])
def test_training_step_with_an_infinite_target(film, channels, freqs):
    log(f"case: training step, FiLM {film}, {channels} channels")
    from tensorf_amd import cameras, render, training
    from tests.test_gpu_mlp_tiles import _reference_layout
    rays, samples, g, ncam = 3, 13, 12, 3
    shape = orc.MlpShape(feat_dim=3 * channels, feature_n_freqs=freqs, viewdir_n_freqs=freqs,
                         num_cameras=ncam if film else None)
    cfg = training.TensorfConfig(
        minibatch_size=rays, n_iters=100, initial_aabb_min=(-1.5,) * 3,
        initial_aabb_max=(1.5,) * 3, appearance_feat_dim=channels, density_feat_dim=16,
        feature_n_freqs=freqs, viewdir_n_freqs=freqs, grid_dim_init=g, grid_dim_final=g,
        upsamp_iters=(), density_samples_per_ray=samples, appearance_samples_per_ray=samples,
        camera_embeddings=film, mlp_precision="fp32", density_shift=-3.0)
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
    colors[1, 0] = np.inf
    batch = cameras.RenderedRays(dev(colors), cameras.Rays3D(dev(o), dev(d),
                                                             dev(cams, torch.int32)))
    jit = render.uniform(render._seed(render._seed(st.prng_key, 0), 1),
                         samples).cpu().numpy().astype(np.float64)
    st.training_step(batch)
    got = _reference_layout(st.flat, st.flat.exp_avg)
    ocfg = orc.RenderConfig(0.05, 200.0, orc.RGB, samples, samples, density_shift=-3.0)
    out, cache = orc.render_rays(p, np.array([[-1.5] * 3, [1.5] * 3]), o, d, cams, ocfg, shape, jit)
    assert _clear(cache["mlp"])[samples:2 * samples].all() and cache["w"].min() > 1e-6
    with np.errstate(invalid="ignore"):
        up = 2.0 * (out - colors) / out.size
        dc = (cache["unbias"][:, None] * cache["wsel"])[:, :, None] * up[:, None, :]
    want, _ = _backward(p, cache["mlp"], dc.reshape(-1, 3), shape)
    for key in KEYS[:len(KEYS) if film else -1]:
        _check(key, 10.0 * got[key], want[key])
