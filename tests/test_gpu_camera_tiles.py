"""The camera embedding's gradient where a tile of the MLP backward (32 rows in FP32,
64 in BF16) holds rays of several cameras: rays of sample counts that do and do not
divide a tile, against the oracle; and the backward takes as long per row as where
tiles lie within a ray (128 samples), though every ray has another camera than its
neighbours (an add per row for such tiles took six times as long with rays of 96
samples and five cameras)."""
import pytest
import torch

from tests import test_gpu_mlp_tiles as tiles
from tests.gpu_common import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("rays,samples", [(3, 96), (5, 45), (9, 16), (17, 5), (40, 2), (70, 1)])
def test_gradient(rays, samples, precision, channels, freqs):
    tiles.test_train_step_gradient_at_tile_edges(rays, samples, precision, True, channels, freqs)


@pytest.mark.parametrize("channels,freqs", [(48, 2), (24, 6)])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_time_per_row(precision, channels, freqs):
    from oracle import tensorf_oracle as orc
    from tensorf_amd import _lib, cameras, training

    def ns_per_row(rays, samples):
        cfg = training.TensorfConfig(
            minibatch_size=rays, n_iters=100, initial_aabb_min=(-1.5,) * 3,
            initial_aabb_max=(1.5,) * 3, appearance_feat_dim=channels, density_feat_dim=16,
            feature_n_freqs=freqs, viewdir_n_freqs=freqs, grid_dim_init=32, grid_dim_final=32,
            upsamp_iters=(), density_samples_per_ray=samples, appearance_samples_per_ray=samples,
            camera_embeddings=True, mlp_precision=precision)
        st = training.TrainState.initialize(cfg, 32, prng_key=3, num_cameras=5)
        o, d = orc.make_rays(rays, seed=8, radius=4.0, target_half=0.5)
        to = lambda a: torch.tensor(a, dtype=torch.float32, device="cuda")
        cams = (torch.arange(rays, device="cuda") % 5).to(torch.int32)
        batch = cameras.RenderedRays(torch.full((rays, 3), 0.5, device="cuda"),
                                     cameras.Rays3D(to(o), to(d), cams))
        for _ in range(3):
            st.training_step(batch)
        torch.cuda.synchronize()
        _lib.profile_enable(True)
        for _ in range(10):
            st.training_step(batch)
        torch.cuda.synchronize()
        ms, launches = _lib.profile_read()["mlp_bwd"]
        _lib.profile_enable(False)
        return 1e6 * ms / launches / (rays * samples)

    whole, mixed = ns_per_row(1536, 128), ns_per_row(2048, 96)
    log(f"  {precision}, {channels} channels: 128 samples {whole:.3f} ns a row, 96 {mixed:.3f}")
    assert mixed < 1.5 * whole
