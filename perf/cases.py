"""Performance cases of the TensoRF render and training path.

Each case is one call a user's program makes through the package's public entry
points, at a size of the configurations this repository names (the reference's
defaults, the benchmark's workloads) or between them:

  train   TrainState.training_step on one minibatch, in the middle of training
  render  render_rays on one chunk of rays (RGB or a distance), no gradients
  grad    render_rays with the gradients of a loss of the program's own
  mlp     FeatureMlp.apply on rows of features, with its backward
  interp  TensorVM.interpolate at points, with its backward

The scene is a smooth random density (a coarse grid interpolated up, as a
trained field is smooth, with a little noise per texel) thresholded at -10, so
that rays cross empty space, surfaces and what lies behind them.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensorf-jax_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

SQUASH, UNITS, CAMERAS = 27, 128, 100
STEP = 5000            # training steps taken before the measured one
NEAR, FAR = 0.05, 200.0
SHIFT = -10.0
PROP0, PROP1, PROP_GRID, PROP_CH, PROP_PAD = 128, 64, 64, 8, 0.64

# The reference's default channels and frequencies, and the benchmark's.
DEFAULTS = dict(cd=8, ca=24, freqs=6)
WIDE = dict(cd=16, ca=48, freqs=2)


def _field(kind, rays, grid, samples, shaded, precision="fp32", contraction=False, cameras=False,
           proposal=False, mode="rgb", cd=16, ca=48, freqs=2):
    return dict(kind=kind, rays=rays, grid=grid, samples=samples, shaded=shaded,
                precision=precision, contraction=contraction, cameras=cameras, proposal=proposal,
                mode=mode, cd=cd, ca=ca, freqs=freqs)


def listed():
    return [
        # a viewer's preview tile while the default configuration trains at its first grid
        dict(_field("render", 1024, 128, 221, 33, **DEFAULTS), name="render_preview_default"),
        # the default configuration's training step at its first grid (sqrt(3) G samples, 15% shaded)
        dict(_field("train", 4096, 128, 221, 33, **DEFAULTS), name="train_default_g128"),
        # and at its last, where most of its 30,000 steps are taken
        dict(_field("train", 4096, 300, 519, 77, **DEFAULTS), name="train_default_g300"),
        # the headline: every one of 512 stratified samples shaded, FP32
        dict(_field("train", 4096, 300, 512, 512, **WIDE), name="train_uniform512_fp32"),
        # proposal sampling with the BF16 MLP: the fast configuration
        dict(_field("train", 16384, 300, 64, 64, "bf16", proposal=True, **WIDE),
             name="train_proposal64_bf16"),
        # per-ray top-64 of 512 samples, BF16 MLP
        dict(_field("train", 8192, 300, 512, 64, "bf16", **WIDE), name="train_top64_bf16"),
        # unbounded scene: contraction, fisheye rays, camera embedding; the largest step
        dict(_field("train", 8192, 300, 512, 512, "bf16", contraction=True, cameras=True, **WIDE),
             name="train_contracted_film_bf16"),
        # one chunk of an 800x800 frame with the proposal sampler
        dict(_field("render", 65536, 300, 64, 64, "bf16", proposal=True, **WIDE),
             name="render_frame_proposal_bf16"),
        # one chunk of a frame's median distances
        dict(_field("render", 65536, 300, 512, 512, mode="median", **WIDE),
             name="render_frame_depth"),
        # a training loop of the program's own (its loss, its optimizer): odd sizes
        dict(_field("grad", 1000, 199, 301, 301, **WIDE), name="grad_own_loss_fp32"),
        # the feature MLP as a layer, ragged row count
        dict(kind="mlp", rows=100003, ca=48, freqs=2, precision="fp32", cameras=False,
             name="mlp_layer_fp32"),
        # feature lookups at points of the program's own (a mesh, an occupancy test)
        dict(kind="interp", points=250001, grid=300, ca=48, name="vm_interpolate_points"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "render", "render", "grad", "mlp", "interp"])
    if kind == "mlp":
        wide = rng.random() < 0.7
        return dict(kind="mlp", rows=_log_int(rng, 500, 500000), ca=48 if wide else 24,
                    freqs=2 if wide else 6, precision=rng.choice(["fp32", "bf16"]),
                    cameras=rng.random() < 0.3)
    if kind == "interp":
        return dict(kind="interp", points=_log_int(rng, 1000, 1000000),
                    grid=_log_int(rng, 64, 300), ca=rng.choice([8, 16, 24, 48]))
    grid = _log_int(rng, 64, 300)
    shape = WIDE if rng.random() < 0.7 else DEFAULTS
    precision = rng.choice(["fp32", "bf16"])
    proposal = kind != "grad" and shape is WIDE and rng.random() < 0.35
    contraction = not proposal and rng.random() < 0.3
    if proposal:
        samples = shaded = rng.choice([48, 64, 96, 128])
    else:
        samples = _log_int(rng, 96, 600)
        share = rng.choice(["all", "top64", "15%"]) if shape is WIDE else "15%"
        shaded = {"all": samples, "top64": min(64, samples), "15%": max(1, int(0.15 * samples))}[share]
    mode = "rgb"
    if kind == "render":
        mode = rng.choice(["rgb", "rgb", "median", "mean"])
        most = min(65536, 4000000 // (shaded if mode == "rgb" else 64))
    elif kind == "grad":
        most = min(8192, 600000 // shaded)
    else:
        most = min(16384, 1500000 // shaded)
    return _field(kind, _log_int(rng, 256, most), grid, samples, shaded, precision, contraction,
                  kind == "train" and rng.random() < 0.3, proposal, mode, **shape)


# ---- inputs --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _factors(g, grid, ch, smooth, noise, coarse=12):
    """Channel-last plane (3, G, G, C) and line (3, G, C)."""
    import torch.nn.functional as F
    plane = F.interpolate(_randn(g, 3, ch, coarse, coarse) * smooth, size=(grid, grid),
                          mode="bilinear", align_corners=True)
    line = F.interpolate(_randn(g, 3, ch, coarse) * smooth, size=grid, mode="linear",
                         align_corners=True)
    plane = plane.permute(0, 2, 3, 1).contiguous()
    line = line.permute(0, 2, 1).contiguous()
    return plane + noise * _randn(g, *plane.shape), line + noise * _randn(g, *line.shape)


def _mlp_leaves(g, ca, freqs, cameras):
    e = SQUASH + 3 + 2 * freqs * SQUASH + 2 * freqs * 3
    f = 3 * ca
    n = lambda i, o, s: _randn(g, i, o) * math.sqrt(s / i)  # noqa: E731
    out = {"w0": n(f, SQUASH, 1), "w1": n(e, UNITS, 2), "b1": 0.1 * _randn(g, UNITS),
           "w2": n(UNITS, UNITS, 2), "b2": 0.1 * _randn(g, UNITS), "w3": n(UNITS, 3, 1),
           "b3": 0.1 * _randn(g, 3)}
    if cameras:
        out["embed"] = torch.cat([1 + 0.1 * _randn(g, CAMERAS, UNITS // 2),
                                  0.1 * _randn(g, CAMERAS, UNITS // 2)], dim=1)
    return out


def _rays(g, case):
    r = case["rays"]
    if case["contraction"]:
        # equidistant fisheye (180 degrees) of cameras on a ring, minibatches shuffled over frames
        cam = torch.randint(0, CAMERAS, (r,), generator=g, device="cuda")
        a = cam.float() * (2 * math.pi / CAMERAS)
        o = torch.stack([3 * torch.cos(a), 3 * torch.sin(a), 0.3 * torch.sin(3 * a)], 1)
        th = torch.rand(r, generator=g, device="cuda").sqrt() * (math.pi / 2)
        ph = torch.rand(r, generator=g, device="cuda") * (2 * math.pi)
        fw = -torch.stack([torch.cos(a), torch.sin(a), torch.zeros_like(a)], 1)
        rt = torch.stack([-torch.sin(a), torch.cos(a), torch.zeros_like(a)], 1)
        up = torch.tensor([0.0, 0.0, 1.0], device="cuda").expand_as(fw)
        d = torch.cos(th)[:, None] * fw + torch.sin(th)[:, None] * (
            torch.cos(ph)[:, None] * rt + torch.sin(ph)[:, None] * up)
    else:
        cam = torch.randint(0, CAMERAS, (r,), generator=g, device="cuda")
        v = _randn(g, r, 3)
        v[:, 2] = v[:, 2].abs()
        o = 4 * v / v.norm(dim=1, keepdim=True)
        d = (torch.rand((r, 3), generator=g, device="cuda") * 2 - 1) * 0.8 - o
        d = d / d.norm(dim=1, keepdim=True)
    return o.contiguous(), d.contiguous(), cam.to(torch.int32)


def _moments(g, leaf, scale):
    """Adam moments of a parameter whose gradients are of size `scale`."""
    m = 0.3 * scale * _randn(g, *leaf.shape)
    v = (scale * (0.5 + torch.rand(leaf.shape, generator=g, device="cuda"))) ** 2
    return m, v


def _inputs(case, seed):
    """Every input of a train, render or grad case, in float32: leaves (name -> tensor in the
    state's layout and order), moments, rays and colours."""
    g = _gen(seed)
    cd, ca = case["cd"], case["ca"]
    leaves = {}
    leaves["density_plane"], leaves["density_line"] = _factors(
        g, case["grid"], cd, math.sqrt(14.8 / math.sqrt(3 * cd)), 0.02)
    leaves["appearance_plane"], leaves["appearance_line"] = _factors(g, case["grid"], ca, 0.6, 0.05)
    leaves.update(_mlp_leaves(g, ca, case["freqs"], case["cameras"]))
    prop = {}
    if case["proposal"]:
        prop["prop_plane"], prop["prop_line"] = _factors(g, PROP_GRID, PROP_CH, 0.8, 0.02)
        f = 3 * PROP_CH
        prop.update(w1=_randn(g, f, 64) / math.sqrt(f), b1=0.1 * _randn(g, 64),
                    w2=_randn(g, 64, 64) / 8, b2=0.1 * _randn(g, 64), w3=_randn(g, 64, 1) / 4,
                    b3=_randn(g, 1) - 1)
    o, d, cam = _rays(g, case)
    colors = torch.rand((case["rays"], 3), generator=g, device="cuda")
    moments = {}
    if case["kind"] == "train":
        for group, tensors in (("", leaves), ("prop.", prop)):
            for name, t in tensors.items():
                moments[group + name] = _moments(g, t, 1e-5 if t.dim() > 2 else 1e-3)
    return dict(leaves=leaves, prop=prop, o=o, d=d, cam=cam, colors=colors, moments=moments)


def _box(case):
    h = 2.0 if case["contraction"] else 1.5
    return [[-h] * 3, [h] * 3]


def _mlp_params(leaves):
    p = {"Dense_0": {"kernel": leaves["w0"]},
         "Dense_1": {"kernel": leaves["w1"], "bias": leaves["b1"]},
         "Dense_2": {"kernel": leaves["w2"], "bias": leaves["b2"]},
         "Dense_3": {"kernel": leaves["w3"], "bias": leaves["b3"]}}
    if "embed" in leaves:
        p["Embed_0"] = {"embedding": leaves["embed"]}
    return {"params": p}


def _proposal_config(case):
    from tensorf_amd import proposal
    return proposal.ProposalConfig(samples_round0=PROP0, samples_round1=PROP1,
                                   samples_out=case["samples"], histogram_pad=PROP_PAD,
                                   grid_dim=PROP_GRID, channels=PROP_CH) \
        if case["proposal"] else None


def _train_state(case, x):
    from tensorf_amd import training
    cfg = training.TensorfConfig(
        minibatch_size=case["rays"], n_iters=30000,
        optimizer=training.OptimizerConfig(lr_init_tensor=0.002, lr_init_mlp=1e-4),
        initial_aabb_min=tuple(_box(case)[0]), initial_aabb_max=tuple(_box(case)[1]),
        appearance_feat_dim=case["ca"], density_feat_dim=case["cd"],
        feature_n_freqs=case["freqs"], viewdir_n_freqs=case["freqs"], upsamp_iters=(),
        scene_contraction=case["contraction"], camera_embeddings=case["cameras"],
        render_near=NEAR, render_far=FAR, density_samples_per_ray=case["samples"],
        appearance_samples_per_ray=case["shaded"], mlp_precision=case["precision"],
        proposal=_proposal_config(case), density_shift=SHIFT)
    state = training.TrainState.initialize(cfg, 16, prng_key=0, num_cameras=CAMERAS)
    state = state.resize_grid(case["grid"])
    for flat, tensors, group in ((state.flat, x["leaves"], ""), (state.prop_flat, x["prop"], "prop.")):
        for i, (name, t) in enumerate(tensors.items()):
            flat.view(flat.params, i).copy_(t)
            flat.view(flat.exp_avg, i).copy_(x["moments"][group + name][0])
            flat.view(flat.exp_avg_sq, i).copy_(x["moments"][group + name][1])
    state.step = state.adam_count = STEP
    return state


def prepare(case, seed):
    from tensorf_amd import cameras, networks, proposal, render, tensor_vm
    if case["kind"] == "interp":
        g = _gen(seed)
        plane, line = _factors(g, case["grid"], case["ca"], 0.6, 0.05)
        ijk = torch.rand((3, case["points"]), generator=g, device="cuda") * 2 - 1
        up = _randn(g, 3 * case["ca"], case["points"])
        vm = tensor_vm.TensorVM(tensor_vm.TensorVMSingle(plane.requires_grad_(True),
                                                         line.requires_grad_(True)))
        return dict(kind="interp", vm=vm, ijk=ijk, up=up)
    if case["kind"] == "mlp":
        x = _mlp_inputs(case, seed)
        mlp = networks.FeatureMlp(feature_n_freqs=case["freqs"], viewdir_n_freqs=case["freqs"],
                                  num_cameras=CAMERAS if case["cameras"] else None,
                                  precision=case["precision"])
        leaves = {k: t.requires_grad_(True) for k, t in x["leaves"].items()}
        return dict(kind="mlp", mlp=mlp, params=_mlp_params(leaves), leaves=leaves,
                    feats=x["feats"].requires_grad_(True), dirs=x["dirs"],
                    cams=x["cams"] if case["cameras"] else None, up=x["up"])
    x = _inputs(case, seed)
    rays = cameras.Rays3D(x["o"], x["d"], x["cam"])
    if case["kind"] == "train":
        return dict(kind="train", state=_train_state(case, x),
                    batch=cameras.RenderedRays(x["colors"], rays))
    leaves = x["leaves"]
    if case["kind"] == "grad":
        leaves = {k: t.requires_grad_(True) for k, t in leaves.items()}
    vm = lambda t, n: tensor_vm.TensorVM(tensor_vm.TensorVMSingle(t[n + "_plane"], t[n + "_line"]))  # noqa: E731
    field = None
    if case["proposal"]:
        field = proposal.ProposalField(vm(x["prop"], "prop"),
                                       {k: x["prop"][k] for k in proposal.MLP_KEYS})
    lp = render.LearnableParams(_mlp_params(leaves), vm(leaves, "appearance"),
                                vm(leaves, "density"), case["contraction"], field)
    mlp = networks.FeatureMlp(feature_n_freqs=case["freqs"], viewdir_n_freqs=case["freqs"],
                              precision=case["precision"])
    mode = {"rgb": render.RenderMode.RGB, "median": render.RenderMode.DIST_MEDIAN,
            "mean": render.RenderMode.DIST_MEAN}[case["mode"]]
    cfg = render.RenderConfig(NEAR, FAR, mode, case["samples"], case["shaded"],
                              density_shift=SHIFT, proposal=_proposal_config(case))
    return dict(kind=case["kind"], mlp=mlp, lp=lp, aabb=torch.tensor(_box(case), device="cuda"),
                rays=rays, cfg=cfg, leaves=leaves, colors=x["colors"])


def run(s):
    from tensorf_amd import render
    if s["kind"] == "interp":
        single = s["vm"].stacked_single_vm
        out = s["vm"].interpolate(s["ijk"])
        gp, gl = torch.autograd.grad(out, [single.plane, single.line], s["up"])
        return {"features": out.detach(), "plane": gp, "line": gl}
    if s["kind"] == "mlp":
        out = s["mlp"].apply(s["params"], s["feats"], s["dirs"], s["cams"])
        grads = torch.autograd.grad(out, [s["feats"], *s["leaves"].values()], s["up"])
        return dict(zip(["rgb", "feats", *s["leaves"]], [out.detach(), *grads]))
    if s["kind"] == "train":
        state, logs = s["state"].training_step(s["batch"])
        out = {"mse": logs["mse"]}
        if "prop_loss" in logs:
            out["prop_loss"] = logs["prop_loss"]
        for flat, group in ((state.flat, ""), (state.prop_flat, "prop.")):
            for i, name in enumerate(flat.names if flat else []):
                name = group + name
                out[name] = flat.view(flat.params, i)
                out[name + ".m"] = flat.view(flat.exp_avg, i)
                out[name + ".v"] = flat.view(flat.exp_avg_sq, i)
        return out
    out = render.render_rays(s["mlp"], s["lp"], s["aabb"], s["rays"], 0, s["cfg"])
    if s["kind"] == "render":
        return {"out": out}
    loss = ((out - s["colors"]) ** 2 + 1e-6).sqrt().mean()
    grads = torch.autograd.grad(loss, list(s["leaves"].values()))
    return dict(zip(["out", *s["leaves"]], [out.detach(), *grads]))


def _mlp_inputs(case, seed):
    g = _gen(seed)
    r = case["rows"]
    leaves = _mlp_leaves(g, case["ca"], case["freqs"], case["cameras"])
    d = _randn(g, r, 3)
    return dict(leaves=leaves, feats=0.3 * _randn(g, r, 3 * case["ca"]),
                dirs=d / d.norm(dim=1, keepdim=True),
                cams=torch.randint(0, CAMERAS, (r,), generator=g, device="cuda").to(torch.int32),
                up=_randn(g, r, 3) / r)


# ---- work ----------------------------------------------------------------------------
def _mlp_flops(ca, freqs):
    e = SQUASH + 3 + 2 * freqs * SQUASH + 2 * freqs * 3
    return 2 * (3 * ca * SQUASH + e * UNITS + UNITS * UNITS + UNITS * 3)


def _mlp_count(ca, freqs, cameras):
    return _mlp_flops(ca, freqs) // 2 + 2 * UNITS + 3 + (CAMERAS * UNITS if cameras else 0)


def work(case):
    if case["kind"] == "interp":
        c, g, m = case["ca"], case["grid"], case["points"]
        fac = 3 * c * g * (g + 1) * 4
        # points in, features out, their gradient in, the factors in and their gradients out
        return {"bytes": m * (12 + 2 * 12 * c) + 2 * fac, "flops": m * 3 * c * 40}
    if case["kind"] == "mlp":
        m, f = case["rows"], 3 * case["ca"]
        p = _mlp_count(case["ca"], case["freqs"], case["cameras"])
        return {"bytes": m * (2 * 4 * f + 12 + 24) + 8 * p,
                "flops": 3 * m * _mlp_flops(case["ca"], case["freqs"])}
    r, n, k, g = case["rays"], case["samples"], case["shaded"], case["grid"]
    rgb = case["mode"] == "rgb"
    count = 3 * g * (g + 1) * (case["cd"] + (case["ca"] if rgb else 0))
    if rgb:
        count += _mlp_count(case["ca"], case["freqs"], case["cameras"])
    # interpolation: a multiply and an add per tap and channel, and the product
    flops = r * n * (3 * case["cd"] * 14 + 60)
    if rgb:
        flops += r * k * (3 * case["ca"] * 14 + _mlp_flops(case["ca"], case["freqs"]))
    if case["proposal"]:
        count += 3 * PROP_GRID * (PROP_GRID + 1) * PROP_CH
        flops += r * (PROP0 + PROP1) * (3 * PROP_CH * 14 + 2 * (24 * 64 + 64 * 64 + 64))
    rays = r * 28 + r * (12 if rgb else 4)
    if case["kind"] == "render":
        return {"bytes": 4 * count + rays, "flops": flops}
    if case["kind"] == "grad":
        return {"bytes": 8 * count + rays + 12 * r, "flops": 3 * flops}
    # parameters and both moments, read and written
    return {"bytes": 24 * count + rays, "flops": 3 * flops}


# ---- the same in 64 bits ---------------------------------------------------------------
_M64 = (1 << 64) - 1


def _seed(key, salt):
    return ((int(key) & _M64) * 0x9E3779B97F4A7C15 + salt * 0xBF58476D1CE4E5B9 + 1) & _M64


def _uniform(seed, n):
    """The counter-based generator of the sampling jitter: splitmix64's finaliser."""
    with np.errstate(over="ignore"):
        z = np.arange(n, dtype=np.uint64) * np.uint64(0xD1B54A32D192ED03)
        z += np.uint64((seed * 0x9E3779B97F4A7C15 + 0x632BE59BD9B4E019) & _M64)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
    return torch.tensor((z >> np.uint64(40)).astype(np.float64) / 16777216.0, device="cuda")


def _tap(x, size):
    u = (x + 1) / 2 * (size - 1)
    lo = torch.floor(u)
    w1 = u - lo
    i = lo.clamp(-2, size + 1).long()
    return i.clamp(0, size - 1), (i + 1).clamp(0, size - 1), 1 - w1, w1


def _vm64(plane, line, p):
    """Features (M, 3C) at normalised points p (M, 3)."""
    size, c = plane.shape[1], plane.shape[-1]
    taps = [_tap(p[:, a], size) for a in range(3)]
    out = []
    for m, (v, a, b) in enumerate(((0, 1, 2), (2, 0, 1), (1, 2, 0))):
        (v0, v1, x0, x1), (a0, a1, y0, y1), (b0, b1, z0, z1) = taps[v], taps[a], taps[b]
        pl = plane[m].reshape(size * size, c)
        ln = line[m].index_select(0, v0) * x0[:, None] + line[m].index_select(0, v1) * x1[:, None]
        pv = 0
        for ia, wa in ((a0, y0), (a1, y1)):
            for ib, wb in ((b0, z0), (b1, z1)):
                pv = pv + pl.index_select(0, ia * size + ib) * (wa * wb)[:, None]
        out.append(ln * pv)
    return torch.cat(out, 1)


def _encode(x, freqs):
    y = x[..., None] * (2.0 ** torch.arange(freqs, device=x.device, dtype=x.dtype))
    return torch.cat([torch.sin(y), torch.cos(y)], -1).reshape(x.shape[0], -1)


def _mlp64(w, f, d, cams, freqs):
    h0 = f @ w["w0"]
    x = torch.cat([h0, d, _encode(h0, freqs), _encode(d, freqs)], 1)
    h = torch.relu(torch.relu(x @ w["w1"] + w["b1"]) @ w["w2"] + w["b2"])
    if "embed" in w:
        e = w["embed"].index_select(0, cams)
        half = UNITS // 2
        h = torch.cat([h[:, :half], e[:, :half] * h[:, half:] + e[:, half:]], 1)
    return torch.sigmoid(h @ w["w3"] + w["b3"])


def _segment(o, d, box):
    t = (box[None] - o[:, None]) / (d[:, None] + 1e-8)
    t0 = t.amin(1).amax(1).clamp(min=0.0)
    t1 = t.amax(1).amin(1)
    ok = t0 < t1
    return torch.where(ok, t0, 0.0), torch.where(ok, torch.maximum(t1, t0 + 1e-3), 1e-3)


def _contract(p):
    n = p.abs().amax(-1, keepdim=True)
    return torch.where(n <= 1, p, (2 - 1 / n.clamp(min=1.0)) * p / n.clamp(min=1.0))


def _schedule(n):
    """Distances and steps of the contracted sampler: half linear in [near, near + 1], half out
    to far, in float32 as tables."""
    nc, nf = n // 2, n - n // 2
    s = np.arange(nc, dtype=np.float32) / np.float32(max(nc - 1, 1))
    close = (np.float32(NEAR) * (np.float32(1) - s) + np.float32(NEAR + 1.0) * s).astype(np.float32)
    start = NEAR + 1.0 + 1.0 / nc
    k = 10.0
    far = (1.0 / (1.0 - np.linspace(0.0, 1.0 - 1 / ((FAR - start) / k + 1), nf)) - 1.0) \
        * np.linspace(1.0, k, nf)
    ts = np.concatenate([close, (start + far).astype(np.float32)])
    st = (np.roll(ts, -1) - ts).astype(np.float32)
    st[-1] = st[-2]
    return (torch.tensor(a.astype(np.float64), device="cuda") for a in (ts, st))


def _probabilities(sigma, steps):
    a = sigma * steps
    e = torch.exp(-torch.cumsum(a, 1))
    prev = torch.cat([torch.ones_like(e[:, :1]), e[:, :-1]], 1)
    return e, -torch.expm1(-a) * prev


def _resample(edges, w, count):
    h = w + PROP_PAD / w.shape[1]
    cdf = torch.cat([torch.zeros_like(h[:, :1]), torch.cumsum(h, 1)], 1)
    q = cdf[:, -1:] * (torch.arange(1, count, device=w.device, dtype=w.dtype) / count)
    j = (torch.searchsorted(cdf, q.contiguous(), right=True) - 1).clamp(0, w.shape[1] - 1)
    lo, hi = cdf.gather(1, j), cdf.gather(1, j + 1)
    e0, e1 = edges.gather(1, j), edges.gather(1, j + 1)
    mid = e0 + ((q - lo) / (hi - lo)).clamp(0, 1) * (e1 - e0)
    return torch.cat([edges[:, :1], mid, edges[:, -1:]], 1)


def _interval_loss(fe, fw, pe, pw):
    """mip-NeRF 360's loss of the field's weights over the proposal's bound, summed."""
    total = torch.cat([torch.zeros_like(pw[:, :1]), torch.cumsum(pw, 1)], 1)
    lo = torch.searchsorted(pe[:, 1:].contiguous(), fe[:, :-1].contiguous(), right=True)
    hi = torch.searchsorted(pe[:, :-1].contiguous(), fe[:, 1:].contiguous())
    bound = torch.where(hi > lo, total.gather(1, hi) - total.gather(1, lo.clamp(max=pw.shape[1])), 0.0)
    return ((fw - bound).clamp(min=0) ** 2 / (fw + 1e-7)).sum()


def _render64(case, w, prop, x, rows, jitter, prop_jitter):
    """Output of the rays `rows` in float64, and the proposal's (unscaled) interval loss."""
    box = torch.tensor(_box(case), device="cuda", dtype=torch.float64)
    o, d, cam = x["o"][rows].double(), x["d"][rows].double(), x["cam"][rows].long()
    r, n, k = o.shape[0], case["samples"], case["shaded"]
    unit = lambda p: (((p - box[0]) / (box[1] - box[0]) - 0.5) * 2).reshape(-1, 3)  # noqa: E731
    rounds = []
    if case["proposal"]:
        t0, t1 = _segment(o, d, box)
        step = (t1 - t0) / PROP0
        edges = t0[:, None] + torch.arange(PROP0 + 1, device="cuda") * step[:, None]
        at = 0
        for count, nxt in ((PROP0, PROP1), (PROP1, n)):
            steps = edges[:, 1:] - edges[:, :-1]
            ts = edges[:, :-1] + prop_jitter[rows, at:at + count] * steps
            f = _vm64(prop["prop_plane"], prop["prop_line"], unit(o[:, None] + ts[..., None] * d[:, None]))
            h = torch.relu(torch.relu(f @ prop["w1"] + prop["b1"]) @ prop["w2"] + prop["b2"])
            sigma = torch.nn.functional.softplus(h @ prop["w3"] + prop["b3"], threshold=1e9)
            pw = _probabilities(sigma.reshape(r, count), steps)[1]
            rounds.append((edges, pw))
            edges = _resample(edges, pw.detach(), nxt)
            at += count
        steps = edges[:, 1:] - edges[:, :-1]
        ts = edges[:, :-1] + jitter[rows] * steps
    elif case["contraction"]:
        base, steps = _schedule(n)
        steps = steps.expand(r, n)
        ts = base + steps * jitter[rows]
    else:
        t0, t1 = _segment(o, d, box)
        steps = ((t1 - t0) / n)[:, None].expand(r, n)
        ts = t0[:, None] + (torch.arange(n, device="cuda") + jitter) * steps
    pts = o[:, None] + ts[..., None] * d[:, None]
    pts = unit(_contract(pts) if case["contraction"] else pts)
    s = _vm64(w["density_plane"], w["density_line"], pts).sum(1) + SHIFT
    sigma = torch.nn.functional.softplus(s, threshold=1e9).reshape(r, n)
    e, wt = _probabilities(sigma, steps)
    last = e[:, -1]
    if case["mode"] == "mean":
        return (wt * ts).sum(1) + last * ts[:, -1], None
    if case["mode"] == "median":
        over = (1 - e) > 0.5
        first = over.float().argmax(1)
        t = torch.where(first == 0, 0.0, ts.gather(1, first[:, None])[:, 0])
        return torch.where(over.any(1), t, math.inf), None
    idx = torch.sort(wt.detach(), dim=1, descending=True, stable=True)[1][:, :k].sort(1)[0] \
        if k < n else torch.arange(n, device="cuda").expand(r, n)
    sel = (idx + torch.arange(r, device="cuda")[:, None] * n).reshape(-1)
    f = _vm64(w["appearance_plane"], w["appearance_line"], pts[sel])
    rgb = _mlp64(w, f, d.repeat_interleave(k, 0), cam.repeat_interleave(k), case["freqs"])
    ws = wt.gather(1, idx)
    unbias = (1 - last + 1e-8) / (ws.sum(1) + 1e-8)
    out = (rgb.reshape(r, k, 3) * ws[..., None]).sum(1) * unbias[:, None] + last[:, None]
    loss = sum(_interval_loss(edges, wt.detach(), pe, pw) for pe, pw in rounds) if rounds else None
    return out, loss


def _adam64(p, g, m, v, lr):
    m = 0.1 * g + 0.9 * m.double()
    v = 0.01 * g * g + 0.99 * v.double()
    c = STEP + 1
    step = m / (1 - 0.9 ** c) / (torch.sqrt(v / (1 - 0.99 ** c)) + 1e-8)
    return p.detach() - lr * step, m, v


def exact(case, seed):
    if case["kind"] == "interp":
        g = _gen(seed)
        plane, line = (t.double().requires_grad_(True)
                       for t in _factors(g, case["grid"], case["ca"], 0.6, 0.05))
        ijk = torch.rand((3, case["points"]), generator=g, device="cuda") * 2 - 1
        up = _randn(g, 3 * case["ca"], case["points"])
        out = _vm64(plane, line, ijk.T.double())
        gp, gl = torch.autograd.grad(out, [plane, line], up.T.double())
        return {"features": out.detach().T, "plane": gp, "line": gl}
    if case["kind"] == "mlp":
        x = _mlp_inputs(case, seed)
        leaves = {k: t.double().requires_grad_(True) for k, t in x["leaves"].items()}
        f = x["feats"].double().requires_grad_(True)
        out = _mlp64(leaves, f, x["dirs"].double(), x["cams"].long(), case["freqs"])
        grads = torch.autograd.grad(out, [f, *leaves.values()], x["up"].double())
        return dict(zip(["rgb", "feats", *leaves], [out.detach(), *grads]))
    x = _inputs(case, seed)
    train, need = case["kind"] == "train", case["kind"] != "render"
    leaves = {k: t.double().requires_grad_(need) for k, t in x["leaves"].items()}
    prop = {k: t.double().requires_grad_(need) for k, t in x["prop"].items()}
    r, n = case["rays"], case["samples"]
    key = _seed(0, STEP) if train else 0
    jitter = prop_jitter = None
    if case["proposal"]:
        m = PROP0 + PROP1
        if train:
            both = _uniform(key, r * (m + n))
            prop_jitter, jitter = both[:r * m].reshape(r, m), both[r * m:].reshape(r, n)
        else:
            prop_jitter = _uniform(_seed(key, 3), r * m).reshape(r, m)
            jitter = _uniform(_seed(key, 1), r * n).reshape(r, n)
    elif case["contraction"]:
        jitter = _uniform(_seed(key, 1), r * n).reshape(r, n)
    else:
        jitter = _uniform(_seed(key, 1), n)
    outs, mse, ploss = [], 0.0, 0.0
    per = max(1, 262144 // max(n, PROP0 if case["proposal"] else 1))
    for at in range(0, r, per):
        rows = slice(at, min(r, at + per))
        with torch.set_grad_enabled(need):
            out, loss = _render64(case, leaves, prop, x, rows, jitter, prop_jitter)
            outs.append(out.detach())
            if not need:
                continue
            diff = out - x["colors"][rows].double()
            part = (diff ** 2).sum() / (3 * r) if train else torch.sqrt(diff ** 2 + 1e-6).sum() / (3 * r)
            mse += part.detach()
            if loss is not None:
                loss = loss / r
                ploss += loss.detach()
                part = part + loss
            part.backward()
    if not need:
        return {"out": torch.cat(outs)}
    if not train:
        return {"out": torch.cat(outs), **{k: t.grad for k, t in leaves.items()}}
    got = {"mse": mse.reshape(1)}
    if case["proposal"]:
        got["prop_loss"] = ploss.reshape(1)
    decay = max(0.1 ** (STEP / 30000), 0.1)
    for group, tensors in (("", leaves), ("prop.", prop)):
        for i, (name, t) in enumerate(tensors.items()):
            lr = decay * (0.002 if i < (2 if group else 4) else 1e-4)
            p, m, v = _adam64(t, t.grad, *x["moments"][group + name], lr)
            got.update({group + name: p, group + name + ".m": m, group + name + ".v": v})
    return got
