"""The forward of a training step (fpscan_scan_fwd_saved, fpscan_scan_fwd_softplus_saved):
another cache policy, the same arithmetic, so the outputs equal the plain forward's bit for
bit on every kernel it can take; and the same refusals.
"""
import ctypes
import os

import pytest
import torch

import fpscan_amd
from conftest import ROOT
from fpscan_amd import ops
from scan_helpers import DEVICE, bits_equal

gpu = [pytest.mark.gpu,
       pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device (MI355X)")]

# (rows, sub-chunks per row): waves per row 1 (four rows a block, one row a block), 2, 4, 8 and
# 16, the ring depths, short rows (0: a row of half a sub-chunk; around 64 MiB), and tensors on
# both sides of 128 MiB, where keeping ends (a sub-chunk is 1 KiB)
ROWS = [(6, 0), (131071, 0), (131072, 0), (6, 1), (32768, 1), (5, 2), (5, 4), (5, 8), (5, 16),
        (2048, 16), (3, 32), (3, 128), (1024, 128), (1025, 128)]


@pytest.mark.parametrize("softplus", [False, True], ids=["gates", "softplus"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("rows,subs", ROWS, ids=lambda v: str(v))
def test_equals_the_plain_forward(dtype, rows, subs, softplus):
    _equal(dtype, rows, subs, softplus, tiling=0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
def test_equals_the_plain_forward_tiled(dtype):
    _equal(dtype, 37, 64, False, tiling=2)


for _t in (test_equals_the_plain_forward, test_equals_the_plain_forward_tiled):
    _t.pytestmark = getattr(_t, "pytestmark", []) + gpu


def _equal(dtype, rows, subs, softplus, tiling):
    sub = 1024 // torch.empty((), dtype=dtype).element_size()
    L = subs * sub if subs else sub // 2
    gen = torch.Generator(device=DEVICE).manual_seed(rows + subs)
    z = torch.randn((1, rows, L), generator=gen, device=DEVICE)
    first = z.to(dtype) if softplus else torch.sigmoid(3 + z).to(dtype)
    x = torch.randn((1, rows, L), generator=gen, device=DEVICE).to(dtype)
    rate = torch.rand(rows, generator=gen, device=DEVICE)
    out = torch.full_like(x, float("nan"))
    ext = ops._load_extension()
    ops.set_tiling(tiling)
    try:
        if softplus:
            want = fpscan_amd.scan_forward_softplus(first, rate, x)
            ext.fullscan_forward_softplus_saved(first, rate, x, out)
        else:
            want = fpscan_amd.scan_forward(first, x)
            ext.fullscan_forward_saved(first, x, out)
    finally:
        ops.set_tiling(0)
    assert bits_equal(out, want)


def test_refuses_what_the_plain_forward_refuses():
    lib = ctypes.CDLL(os.path.join(ROOT, "fpscan_amd", "libfpscan_hip.so"))
    vp, i64, c_int = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    lib.fpscan_scan_fwd.argtypes = [vp, vp, vp, i64, i64, i64, i64, i64, c_int, c_int, vp,
                                    ctypes.c_size_t, vp]
    lib.fpscan_scan_fwd_saved.argtypes = [vp, vp, vp, i64, i64, i64, i64, i64, c_int, vp,
                                          ctypes.c_size_t, vp]
    p = 4096  # never dereferenced: each call is refused, or has nothing to do
    for ptrs, shape, dtype in [((p, p, p), (1, 1, 48, 48, 48), 0), ((p, p, p), (1, 1, 64, 64, 64), 7),
                               ((p, p, None), (1, 1, 64, 64, 64), 0), ((p, p + 4, p), (1, 1, 64, 64, 64), 0),
                               ((p, p, p), (2, 2, 64, 128, 63), 0), ((p, p, p), (0, 4, 64, 256, 64), 2)]:
        want = lib.fpscan_scan_fwd(*ptrs, *shape, dtype, 0, None, 0, None)
        assert lib.fpscan_scan_fwd_saved(*ptrs, *shape, dtype, None, 0, None) == want
