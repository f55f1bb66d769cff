"""The sort of (row, mode) pairs counts three pairs a row in 32-bit signed
integers: a batch of more rows than that is not sorted (the direct scatter
takes it), in the render backward and in the interpolation backward. Checked on
the CPU: the rule of the render backward from a host program built from the
header, that of the interpolation backward from its workspace size."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LAST = (2 ** 31 - 1) // 3  # the most rows whose pairs an int32 counts
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROBE = r"""
#include <stdio.h>
#include <stdlib.h>
#include "tfh_scatter_sorted.h"
int main(int argc, char** argv) {
  float f = 0;
  uint32_t order = 0;
  tfh::SortWs s;
  s.order = &order;
  for (int i = 1; i < argc; ++i)
    for (int64_t channels : {1, 8, 16, 48, 64})
      printf("%d ", (int)tfh::sorted_scatter_ok(tfh_vm{&f, &f, 300, channels}, atoll(argv[i]), s));
}
"""


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
def test_render_scatter_sorts_no_more_pairs_than_it_counts(tmp_path):
    src, exe = tmp_path / "probe.hip", tmp_path / "probe"
    src.write_text(PROBE)
    csrc = os.path.join(ROOT, "tensorf-jax_amd", "csrc")
    lib = os.path.join(ROOT, "tensorf-jax_amd", "tensorf_amd", "libtensorf_hip.so")
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-I" + csrc,
                    "-I" + os.path.join(ROOT, "include"), str(src), "-c", "-o",
                    str(tmp_path / "probe.o")], check=True, capture_output=True)
    subprocess.run([HIPCC, str(tmp_path / "probe.o"), lib, "-o", str(exe)], check=True,
                   capture_output=True)
    rows = [1, LAST, LAST + 1, 2 ** 30 - 1, 2 ** 30, 2 ** 40]
    out = subprocess.run([str(exe), *map(str, rows)], check=True, capture_output=True, text=True,
                         env={**os.environ, "LD_LIBRARY_PATH": os.path.dirname(lib) + ":" +
                              os.environ.get("LD_LIBRARY_PATH", "")})
    got = [int(v) for v in out.stdout.split()]
    assert got == [int(m <= LAST) for m in rows for _ in range(5)]


@pytest.mark.parametrize("channels", [1, 8, 16, 48, 64])
def test_interpolation_sorts_no_more_pairs_than_it_counts(channels):
    from tensorf_amd import _lib
    vm = _lib.Vm(256, 256, 300, channels)  # (never read: a size query)

    def size(points):
        return _lib.lib.tfh_vm_interpolate_bwd_workspace_size(ctypes.byref(vm), points)

    assert size(1 << 20) > 0
    per_point = 3 * channels * 4 + 30  # a row of gradients and the pairs' sort
    for points in (LAST + 1, 2 ** 30 - 1, 2 ** 30):
        # either not sorted at once or not sorted at all
        assert size(points) <= LAST * per_point + (1 << 20)
