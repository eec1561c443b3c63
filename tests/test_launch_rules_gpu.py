"""The automatic launch shapes of the row-streaming kernels at the sizes where their rules
change, against the oracle on sampled rows (every shape itself is forced in
test_scan_gpu.test_every_launch_shape)."""
import pytest
import torch

import fpscan_amd
import oracle
from scan_helpers import DEVICE, check

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device (MI355X)"),
]

# (rows, sub-chunks per row): the plain backward's 8 waves from 16 MiB (and just below) to 128
# MiB (and just above), on the longest rows (256 fp32 sub-chunks, 128 of a 2-byte type)
EIGHT = [(16 * 8 - 1, 128), (16 * 8, 128), (1024, 128), (1025, 128)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("rows,subs", EIGHT, ids=str)
def test_long_rows_backward(dtype, rows, subs):
    _check(dtype, rows, subs)


def _check(dtype, rows, subs):
    L = subs * (1024 // torch.empty((), dtype=dtype).element_size())
    gen = torch.Generator(device=DEVICE).manual_seed(rows)
    g = torch.sigmoid(3 + torch.randn((1, rows, L), generator=gen, device=DEVICE)).to(dtype)
    x, go = (torch.randn((1, rows, L), generator=gen, device=DEVICE).to(dtype) for _ in range(2))
    y = fpscan_amd.scan_forward(g, x)
    gg, gx = fpscan_amd.scan_backward(g, y, go)
    pick = torch.tensor(sorted({0, 1, rows // 2, rows - 2, rows - 1}))
    at = [t[:, pick].cpu() for t in (g, x, go, y, gg, gx)]
    check(at[3], oracle.scan_f64(at[0], at[1]), dtype, "forward")
    gg_ref, gx_ref = oracle.scan_bwd_f64(at[0], at[3], at[2])
    check(at[5], gx_ref, dtype, "grad_tokens")
    check(at[4], gg_ref, dtype, "grad_gates")
    assert torch.isfinite(gg).all() and torch.isfinite(gx).all()
