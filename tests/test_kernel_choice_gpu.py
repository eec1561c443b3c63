"""Which kernel a call launches, by the name that the profiler records: the rules that give the same
results either way and would otherwise show only in the time.
"""
import re

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

import fpscan_amd
import oracle
from scan_helpers import DEVICE, check

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device (MI355X)"),
]


def kernels(call):
    """(kernel name, template arguments) of the scan kernels that ``call`` launches, in order."""
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    found = []
    for event in prof.events():
        m = re.search(r"(scan_\w+|clear_status)(?:<(.*)>)?\(", event.name)
        if m and event.device_type == torch.autograd.DeviceType.CUDA:
            found.append((m[1], re.sub(r"\(anonymous namespace\)::", "", m[2] or "").split(", ")))
    assert found, "the profiler saw no kernel of the library"
    return found


# scan_long_rows<type, mode, waves, sub-chunks in flight, gates, rows per block, cache policy>
@pytest.mark.parametrize("subs,mib,fwd_waves,bwd_waves", [(8, 7, 8, 8), (8, 8, 4, 4), (4, 7, 4, 4),
                                                          (4, 8, 2, 4)], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
def test_waves_of_softplus_rows_of_four_and_eight_sub_chunks(dtype, subs, mib, fwd_waves, bwd_waves):
    L = subs * (1024 // torch.empty((), dtype=dtype).element_size())
    z = torch.randn((1, mib * 1024 // subs, L), device=DEVICE).to(dtype)
    rate = torch.rand(z.shape[1], device=DEVICE)
    for reverse in (False, True):
        (name, args), = kernels(lambda: fpscan_amd.scan_forward_softplus(z, rate, z, reverse))
        assert (name, args[2]) == ("scan_long_rows", str(fwd_waves))
    (name, args), = kernels(lambda: fpscan_amd.scan_backward_softplus(z, rate, z, z))
    assert (name, args[2]) == ("scan_long_rows", str(bwd_waves))


# the backward takes 8 waves on rows of any length from 16 to 128 MiB after a saved forward, from 256
# rows; on its own only on rows of 16 to 64 sub-chunks up to 64 MiB (a sub-chunk is 1 KiB)
@pytest.mark.parametrize("rows,subs,alone,after", [(256, 128, 16, 8), (255, 128, 16, 16),
                                                   (1024, 128, 16, 8), (1025, 128, 16, 16),
                                                   (1024, 16, 8, 8), (1023, 16, 16, 16),
                                                   (4096, 32, 16, 8)], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
def test_waves_of_the_backward(dtype, rows, subs, alone, after):
    shape = (1, rows, subs * (1024 // torch.empty((), dtype=dtype).element_size()))
    g = torch.sigmoid(3 + torch.randn(shape, device=DEVICE)).to(dtype)
    x, go = (torch.randn(shape, device=DEVICE).to(dtype) for _ in range(2))
    y = fpscan_amd.scan_forward(g, x)
    (name, args), = kernels(lambda: fpscan_amd.scan_backward(g, y, go))
    assert (name, args[2]) == ("scan_long_rows", str(alone))
    for apply in (fpscan_amd.pscan, fpscan_amd.PScan.apply):
        leaves = [t.clone().requires_grad_() for t in (g, x)]
        out = apply(*leaves)
        (name, args), = kernels(lambda: out.backward(go))
        assert (name, args[2]) == ("scan_long_rows", str(after))
        pick = [0, rows - 1]
        gg_ref, gx_ref = oracle.scan_bwd_f64(g[:, pick].cpu(), out[:, pick].detach().cpu(),
                                             go[:, pick].cpu())
        check(leaves[0].grad[:, pick].cpu(), gg_ref, dtype, "grad_gates")
        check(leaves[1].grad[:, pick].cpu(), gx_ref, dtype, "grad_tokens")


# the last template argument of scan_long_rows and scan_cl_blocks is the cache policy, 0 if streamed
@pytest.mark.parametrize("name,shape", [("pscan", (2, 64, 4096)), ("pscan_channel_last", (2, 2048, 256)),
                                        ("pscan_softplus", (2, 64, 4096))])
def test_a_forward_that_autograd_does_not_record_streams(name, shape):
    make = lambda *s: torch.rand(s, device=DEVICE, requires_grad=True)  # noqa: E731
    inputs = [make(*shape), make(*shape)]
    if name == "pscan_softplus":
        inputs.insert(1, make(shape[1]))
    call = getattr(fpscan_amd, name)
    policy = lambda f: kernels(f)[-1][1][-1]  # noqa: E731
    assert policy(lambda: call(*inputs)) != "0"
    with torch.no_grad():
        assert policy(lambda: call(*inputs)) == "0"
        assert not call(*inputs).requires_grad
    plain = [t.detach() for t in inputs]
    assert policy(lambda: call(*plain)) == "0"
    for i in range(len(inputs)):  # any one of them is enough
        one = [t.requires_grad_() if i == j else t for j, t in enumerate(t.detach() for t in inputs)]
        assert policy(lambda: call(*one)) != "0"


# scan_cl_blocks<type, mode, steps a lane, cache policy>: the backward on the 128-byte lines (chains of
# 8 vectors) takes 8 steps a lane where one tile of 256 steps holds a sequence of more than 128, and
# from 12 such tiles below 128 chains
@pytest.mark.parametrize("seqlen,chains,steps", [(128, 3, 4), (129, 3, 8), (256, 3, 8), (257, 3, 4),
                                                 (128, 60, 4), (256, 60, 8), (257, 60, 4),
                                                 (3071, 20, 4), (3072, 20, 8), (3072, 127, 8),
                                                 (3072, 128, 4)], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
def test_steps_of_the_channel_last_backward(dtype, seqlen, chains, steps):
    shape = (1, seqlen, chains * 128 // torch.empty((), dtype=dtype).element_size())
    g = (0.9 + 0.09 * torch.rand(shape, device=DEVICE)).to(dtype)
    y, go = (torch.randn(shape, device=DEVICE).to(dtype) for _ in range(2))
    run = lambda: fpscan_amd.scan_backward_channel_last(g, y, go)  # noqa: E731
    name, args = kernels(run)[-1]
    assert (name, args[2]) == ("scan_cl_blocks", str(steps))
    gg, gx = run()
    pick = [0, 1, shape[2] - 1]
    gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(*(t[..., pick].cpu() for t in (g, y, go)))
    check(gx[..., pick].cpu(), gx_ref, dtype, "grad_tokens")
    check(gg[..., pick].cpu(), gg_ref, dtype, "grad_gates")


# off the lines with enough strips: the forward of rows of 20 to 32 vectors takes the one pass with 576
# to 1024 sequences, blocks around that and on fewer vectors; the backward always blocks
@pytest.mark.parametrize("batch,vectors,fwd", [(575, 21, "scan_cl_blocks"), (576, 20, "scan_cl"),
                                               (1024, 31, "scan_cl"), (1025, 20, "scan_cl_blocks"),
                                               (700, 19, "scan_cl_blocks")], ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
def test_kernel_of_narrow_rows_with_enough_strips(dtype, batch, vectors, fwd):
    shape = (batch, 260, vectors * (16 // torch.empty((), dtype=dtype).element_size()))
    g = (0.9 + 0.09 * torch.rand(shape, device=DEVICE)).to(dtype)
    x, go = (torch.randn(shape, device=DEVICE).to(dtype) for _ in range(2))
    for reverse in (False, True):
        assert kernels(lambda: fpscan_amd.scan_forward_channel_last(g, x, reverse))[-1][0] == fwd
    y = fpscan_amd.scan_forward_channel_last(g, x)
    at = [t[-1:].cpu() for t in (g, x, go, y)]
    check(at[3], oracle.scan_f64_channel_last(at[0], at[1]), dtype, "forward")
    run = lambda: fpscan_amd.scan_backward_channel_last(g, y, go)  # noqa: E731
    assert kernels(run)[-1][0] == "scan_cl_blocks"
    gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(at[0], at[3], at[2])
    gg, gx = run()
    check(gx[-1:].cpu(), gx_ref, dtype, "grad_tokens")
    check(gg[-1:].cpu(), gg_ref, dtype, "grad_gates")


# split rows on 64-byte lines: the fp32 backward with 48 chains (panels of 8 vectors) or more takes the
# ring of tiles from 96 MiB, the forward and fewer chains from 192 MiB
@pytest.mark.parametrize("shape,bwd", [((8, 13107, 240), "scan_cl_blocks"),
                                       ((8, 13108, 240), "scan_cl_tiles"),
                                       ((6, 17477, 240), "scan_cl_tiles"),
                                       ((5, 20972, 240), "scan_cl_blocks")], ids=str)
def test_kernel_of_the_fp32_backward_on_64_byte_lines(shape, bwd):
    g = 0.9 + 0.09 * torch.rand(shape, device=DEVICE)
    x, go = (torch.randn(shape, device=DEVICE) for _ in range(2))
    assert kernels(lambda: fpscan_amd.scan_forward_channel_last(g, x))[-1][0] == "scan_cl_blocks"
    y = fpscan_amd.scan_forward_channel_last(g, x)
    run = lambda: fpscan_amd.scan_backward_channel_last(g, y, go)  # noqa: E731
    assert kernels(run)[-1][0] == bwd
    gg, gx = run()
    at = [t[-1:, :, [0, -1]].cpu() for t in (g, y, go, gg, gx)]
    gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(*at[:3])
    check(at[4], gx_ref, torch.float32, "grad_tokens")
    check(at[3], gg_ref, torch.float32, "grad_gates")
