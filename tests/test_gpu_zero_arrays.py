"""Clearing several arrays in one launch: sizes around a workgroup's chunk, an
array at an odd address, an empty one, and the values next to each untouched."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (3, 16384, 5), (16385, 0, 40000, 16383),
                                   tuple(range(1, 17))])
@pytest.mark.parametrize("shift", [0, 1])
def test_zero_arrays(sizes, shift):
    from tensorf_amd import _lib
    bufs = [torch.ones(n + 8, device="cuda") for n in sizes]
    n = len(sizes)
    _lib.call("tfh_zero_arrays", (_lib.c_p * n)(*[b.data_ptr() + 4 * shift for b in bufs]),
              (_lib.c_i64 * n)(*sizes), n, _lib.stream())
    torch.cuda.synchronize()
    for b, m in zip(bufs, sizes):
        assert b[:shift].eq(1).all() and b[shift + m:].eq(1).all()
        assert b[shift:shift + m].eq(0).all()


def test_zeros_like_keeps_shapes_and_types():
    from tensorf_amd import _lib
    ts = [torch.randn(3, 5, device="cuda"), torch.randn(7, device="cuda")]
    for t, z in zip(ts, _lib.zeros_like(ts)):
        assert z.shape == t.shape and z.eq(0).all() and z.dtype is torch.float32
    with pytest.raises(_lib.TfhError):
        _lib.call("tfh_zero_arrays", None, None, 17, _lib.stream())
