"""The memory of TensorVM.interpolate's backward: its workspace does not grow with
the batch past 4 Mi points, a batch of several parts gives the gradients of the
direct scatter, and without room for the workspace the direct scatter runs.
Gradients to 2e-4 of the largest (the order of the FP32 sums)."""
import ctypes

import numpy as np
import pytest
import torch

from tests.gpu_common import dev, f32, log, report

PART = 1 << 22


@pytest.mark.parametrize("channels", [1, 8, 16, 48, 64])
def test_workspace_is_bounded(channels):
    from tensorf_amd import _lib
    vm = _lib.Vm(256, 256, 300, channels)  # (never read: a size query)

    def size(points):
        return _lib.lib.tfh_vm_interpolate_bwd_workspace_size(ctypes.byref(vm), points)

    most = size(PART)
    assert 0 < size(100000) < most < PART * (12 * channels + 30) + (1 << 20)
    for points in (PART + 1, 3 * PART - 1, 10 ** 9, 2 ** 30, 2 ** 40):
        assert 0 < size(points) <= most


def _case(points, channels, g):
    from tensorf_amd import tensor_vm
    rng = np.random.default_rng(1)
    vm = tensor_vm.TensorVM.from_reference_layout(
        dev(f32(rng.normal(size=(3, channels, g)))), dev(f32(rng.normal(size=(3, channels, g, g)))))
    gen = torch.Generator("cuda").manual_seed(2)
    ijk = 2.2 * torch.rand((3, points), device="cuda", generator=gen) - 1.1
    up = torch.randn((3 * channels, points), device="cuda", generator=gen)
    return vm, ijk, up


def _gradients(vm, ijk, up):
    single = vm.stacked_single_vm
    leaves = [single.plane.requires_grad_(True), single.line.requires_grad_(True)]
    return torch.autograd.grad(vm.interpolate(ijk), leaves, up)


def _direct(vm, ijk, up):
    from tensorf_amd import _lib
    single = vm.stacked_single_vm
    out = [torch.zeros_like(single.plane), torch.zeros_like(single.line)]
    c = _lib.Vm(_lib.ptr(single.plane), _lib.ptr(single.line), single.grid_dim(),
                single.channel_dim())
    g = _lib.VmGrad(_lib.ptr(out[0]), _lib.ptr(out[1]))
    _lib.call("tfh_vm_interpolate_bwd", ctypes.byref(c), _lib.ptr(ijk), ijk.shape[1], _lib.ptr(up),
              ctypes.byref(g), _lib.stream())
    return out


def _same(got, want):
    for name, g, w in zip(("plane", "line"), got, want):
        e = report(name, g.detach().cpu().numpy(), w.detach().cpu().numpy())
        assert e.max() <= 2e-4 * float(w.abs().max()), name


@pytest.mark.gpu
@pytest.mark.parametrize("points,channels", [(PART, 2), (PART + 1, 2), (2 * PART + 7, 3)])
def test_parts(points, channels):
    log(f"case: {points} points, {channels} channels")
    args = _case(points, channels, 300)
    _same(_gradients(*args), _direct(*args))


@pytest.mark.gpu
def test_no_room_for_the_workspace(monkeypatch):
    log("case: no room for the sort")
    vm, ijk, up = _case(90001, 48, 40)
    want = _gradients(vm, ijk, up)
    empty = torch.empty

    def no_room(*args, **kwargs):
        if kwargs.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", no_room)
    got = _gradients(vm, ijk, up)
    monkeypatch.undo()
    _same(got, want)
