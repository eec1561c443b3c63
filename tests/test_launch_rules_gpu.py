"""The automatic launch shapes of the row-streaming kernels at the sizes where their rules
change, against the oracle on sampled rows (every shape itself is forced in
test_scan_gpu.test_every_launch_shape)."""
import pytest
import torch

import fpscan_amd
import oracle
from scan_helpers import DEVICE, NORM_TOL, check

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


# half the waves: the plain forward on rows of 8 sub-chunks from 16 to 256 MiB
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("rows,subs", [(2047, 8), (2048, 8), (32768, 8), (32769, 8)], ids=str)
def test_rows_of_eight_sub_chunks(dtype, rows, subs):
    _check(dtype, rows, subs)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("reverse", [False, True], ids=["fwd", "rev"])
@pytest.mark.parametrize("rows,subs", [(3, 4), (7, 8), (2048, 8)], ids=str)
def test_softplus_rows_of_four_and_eight_sub_chunks(dtype, rows, subs, reverse):
    L = subs * (1024 // torch.empty((), dtype=dtype).element_size())
    gen = torch.Generator(device=DEVICE).manual_seed(rows)
    z, x, go = (torch.randn((1, rows, L), generator=gen, device=DEVICE).to(dtype)
                for _ in range(3))
    rate = 0.1 * torch.rand(rows, generator=gen, device=DEVICE)
    y = fpscan_amd.scan_forward_softplus(z, rate, x, reverse)
    pick = torch.tensor(sorted({0, rows // 2, rows - 1}))
    at = [t[:, pick].cpu() for t in (z, x, go)]
    r = rate[pick].cpu()
    check(y[:, pick].cpu(), oracle.scan_softplus_f64(at[0], r, at[1], reverse), dtype, "forward")
    if not reverse:
        gz, gr, gx = fpscan_amd.scan_backward_softplus(z, rate, y, go)
        gz_ref, gr_ref, gx_ref = oracle.scan_bwd_softplus_f64(at[0], r, y[:, pick].cpu(), at[2])
        check(gz[:, pick].cpu(), gz_ref, dtype, "grad_z")
        check(gx[:, pick].cpu(), gx_ref, dtype, "grad_tokens")
        assert oracle.normwise_error(gr[pick], gr_ref) <= max(NORM_TOL[dtype], 1e-4)  # as test_softplus


# short rows (64 elements): one wave per block from 64 MiB per tensor, a last block that is
# partly empty, and the size just below
@pytest.mark.parametrize("dtype,rows", [(torch.float32, (1 << 18) - 1), (torch.float32, 1 << 18),
                                        (torch.float32, (1 << 18) + 1),
                                        (torch.bfloat16, (1 << 19) - 1),
                                        (torch.bfloat16, (1 << 19) + 5)], ids=str)
def test_short_rows_around_64_mib(dtype, rows):
    _check(dtype, rows, 64 * torch.empty((), dtype=dtype).element_size() / 1024)


# the same kernels with the fused gates, and the plain reverse: the fewest and the most lanes a row (4 and
# 32; fp32 8), rows that leave the last block (16 to 2 rows) partly empty, just below 64 MiB and above
@pytest.mark.parametrize("below", [True, False], ids=["below", "above"])
@pytest.mark.parametrize("dtype,L", [(torch.bfloat16, 32), (torch.float16, 32), (torch.float16, 256),
                                     (torch.float32, 32), (torch.float32, 128)], ids=str)
def test_short_rows_with_fused_gates_and_reverse(dtype, L, below):
    rows = (64 << 20) // (L * torch.empty((), dtype=dtype).element_size()) + (-1 if below else 3)
    gen = torch.Generator(device=DEVICE).manual_seed(rows)
    z, x, go = (torch.randn((1, rows, L), generator=gen, device=DEVICE).to(dtype) for _ in range(3))
    rate = 0.1 * torch.rand(rows, generator=gen, device=DEVICE)
    pick = torch.tensor(sorted({0, 1, rows // 2, *range(rows - 17, rows)}))
    zp, xp, gop, rp = *(t[:, pick].cpu() for t in (z, x, go)), rate[pick].cpu()
    for reverse in (True, False):
        y = fpscan_amd.scan_forward_softplus(z, rate, x, reverse)
        check(y[:, pick].cpu(), oracle.scan_softplus_f64(zp, rp, xp, reverse), dtype, "softplus")
        assert torch.isfinite(y).all()
    gz, gr, gx = fpscan_amd.scan_backward_softplus(z, rate, y, go)
    gz_ref, gr_ref, gx_ref = oracle.scan_bwd_softplus_f64(zp, rp, y[:, pick].cpu(), gop)
    check(gz[:, pick].cpu(), gz_ref, dtype, "grad_z")
    check(gx[:, pick].cpu(), gx_ref, dtype, "grad_tokens")
    assert oracle.normwise_error(gr[pick], gr_ref) <= max(NORM_TOL[dtype], 1e-4)  # as test_softplus
    assert all(torch.isfinite(t).all() for t in (gz, gr, gx))
    y = fpscan_amd.scan_forward(torch.sigmoid(3 + z), x, reverse=True)
    check(y[:, pick].cpu(), oracle.scan_f64(torch.sigmoid(3 + z)[:, pick].cpu(), xp, True), dtype,
          "reverse")


def _check(dtype, rows, subs):
    L = int(subs * (1024 // torch.empty((), dtype=dtype).element_size()))
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
