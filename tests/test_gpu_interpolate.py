"""TensorVM.interpolate at points of the program's own: the values at point counts
around a workgroup's rows, and the factor gradients of many points, which are
sorted by cell, against the sum of few at a time, which are not. Points beyond the
grid and on its edges are among them. Values to 2e-6 of the largest (a dozen FP32
operations), gradients to 2e-4 of the largest (the order of the FP32 sums)."""
import numpy as np
import pytest
import torch

from oracle import tensorf_oracle as orc
from tests.gpu_common import dev, f32, log, report

pytestmark = pytest.mark.gpu


def _factors(c, g, seed):
    rng = np.random.default_rng(seed)
    return f32(rng.normal(size=(3, c, g))), f32(rng.normal(size=(3, c, g, g)))


def _points(m, g, seed):
    rng = np.random.default_rng(seed)
    p = rng.uniform(-1.1, 1.1, (3, m))
    p[:, ::7] = np.round((p[:, ::7] + 1) / 2 * (g - 1)) / (g - 1) * 2 - 1  # texel centres
    return f32(p)


@pytest.mark.parametrize("channels", [1, 4, 8, 12, 20, 48, 64, 18])
@pytest.mark.parametrize("m", [1, 31, 33, 100])
def test_values(m, channels):
    log(f"case: {m} points, {channels} channels")
    from tensorf_amd import tensor_vm
    vec, mat = _factors(channels, 17, 1)
    vm = tensor_vm.TensorVM.from_reference_layout(dev(vec), dev(mat))
    p = _points(m, 17, 2)
    want = orc.vm_interpolate(vec.astype(np.float64), mat.astype(np.float64), p.astype(np.float64),
                              np.float64)
    got = vm.interpolate(dev(p)).cpu().numpy()
    assert report("values", got, want).max() <= 2e-6 * np.abs(want).max()


@pytest.mark.parametrize("channels", [3, 8, 12, 24, 64, 18])
@pytest.mark.parametrize("g", [9, 40])
def test_gradients_of_many_points(g, channels):
    m, part = 90001, 30000
    log(f"case: {m} points, {channels} channels, grid {g}")
    from tensorf_amd import tensor_vm
    vec, mat = _factors(channels, g, 1)
    vm = tensor_vm.TensorVM.from_reference_layout(dev(vec), dev(mat))
    single = vm.stacked_single_vm
    leaves = [single.plane.requires_grad_(True), single.line.requires_grad_(True)]
    p = dev(_points(m, g, 2))
    up = torch.randn((3 * channels, m), device="cuda",
                     generator=torch.Generator(device="cuda").manual_seed(3))

    def gradients(at, n):
        out = vm.interpolate(p[:, at:at + n].contiguous())
        return torch.autograd.grad(out, leaves, up[:, at:at + n].contiguous())

    whole = gradients(0, m)
    sums = [torch.zeros_like(t, dtype=torch.float64) for t in leaves]
    for at in range(0, m, part):
        for s, t in zip(sums, gradients(at, min(part, m - at))):
            s += t.double()
    for name, t, s in zip(("plane", "line"), whole, sums):
        e = report(name, t.cpu().numpy(), s.cpu().numpy())
        assert e.max() <= 2e-4 * float(s.abs().max()), name
