"""pscan_channel_last and pscan_softplus run the extension's C++ autograd functions; their
Python twins (PScanChannelLast, PScanSoftplus) launch the same kernels on the same saved
tensors, so outputs and gradients agree bit for bit. grad_rate is the batch sum of the rows'
partial sums, rounded once from double."""
import pytest
import torch

import fpscan_amd
from fpscan_amd import ops
from scan_helpers import DEVICE, bits_equal

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device (MI355X)"),
]


def _leaves(softplus, dtype, shape):
    gen = torch.Generator(device=DEVICE).manual_seed(11)
    a, x, go = (torch.randn(shape, generator=gen, device=DEVICE) for _ in range(3))
    rate = torch.rand(shape[1], generator=gen, device=DEVICE)
    first = [a.to(dtype), rate] if softplus else [torch.sigmoid(3 + a).to(dtype)]
    return [*first, (0.1 * x).to(dtype)], go.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("softplus", [False, True], ids=["channel_last", "softplus"])
def test_agrees_with_the_python_function(softplus, dtype):
    leaves, go = _leaves(softplus, dtype, (3, 256, 512))
    fns = ((fpscan_amd.pscan_softplus, fpscan_amd.PScanSoftplus.apply) if softplus else
           (fpscan_amd.pscan_channel_last, fpscan_amd.PScanChannelLast.apply))
    results = []
    for fn in fns:
        own = [t.clone().requires_grad_() for t in leaves]
        y = fn(*own)
        # a gradient that is not contiguous
        y.backward(go.transpose(1, 2).contiguous().transpose(1, 2))
        results.append([y.detach()] + [t.grad for t in own])
    for a, b in zip(*results):
        assert bits_equal(a, b)
    own = [t.clone() for t in leaves]
    own[-1].requires_grad_()  # the tokens alone
    (gx,) = torch.autograd.grad(fns[0](*own), (own[-1],), go)
    assert bits_equal(gx, results[0][-1])
    assert not fns[0](*leaves).requires_grad


@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5, 33])
@pytest.mark.parametrize("dim", [1, 63, 64, 65])
def test_rate_gradient_is_the_batch_sum(batch, dim):
    gen = torch.Generator(device=DEVICE).manual_seed(batch * 100 + dim)
    z, x, go = (torch.randn((batch, dim, 64), generator=gen, device=DEVICE) for _ in range(3))
    rate = 0.1 * torch.rand((dim, 1), generator=gen, device=DEVICE)
    out = fpscan_amd.scan_forward_softplus(z, rate, x)
    _, grad_rate, _ = fpscan_amd.scan_backward_softplus(z, rate, out, go)
    rows = torch.empty(batch * dim, device=DEVICE)
    ops._load_extension().fullscan_backward_softplus(z, rate, out, go, torch.empty_like(z),
                                                     torch.empty_like(z), rows)
    assert grad_rate.shape == rate.shape
    want = rows.view(batch, dim).double().sum(0).view(rate.shape)
    # one rounding to fp32, and the double sums' own order
    assert ((grad_rate.double() - want).abs() <= 2.0 ** -24 * want.abs() + 1e-14).all()


# one launch, two with a last slice that is short, and the most slices; channels that fill no wave
@pytest.mark.parametrize("batch,dim", [(512, 64), (513, 64), (513, 65), (40000, 40), (32769, 1),
                                       (100003, 3)], ids=str)
def test_rate_gradient_of_long_batches(batch, dim):
    gen = torch.Generator(device=DEVICE).manual_seed(batch)
    rate = 0.1 * torch.rand(dim, generator=gen, device=DEVICE)
    z, x, go = (torch.randn((batch, dim, 32), generator=gen, device=DEVICE) for _ in range(3))
    rows = torch.empty(batch * dim, device=DEVICE)
    ops._load_extension().fullscan_backward_softplus(z, rate, x, go, torch.empty_like(z),
                                                     torch.empty_like(z), rows)
    _, grad_rate, _ = fpscan_amd.scan_backward_softplus(z, rate, x, go)
    rows = rows.view(batch, dim).double()
    # one rounding to fp32, and the double sums' own order
    bound = 2.0 ** -24 * rows.sum(0).abs() + batch * 2.0 ** -52 * rows.abs().sum(0)
    assert ((grad_rate.double() - rows.sum(0)).abs() <= bound).all()


def test_rate_gradient_of_a_long_batch_costs_less_than_the_scan():
    z, out, go = (torch.randn((65536, 64, 32), device=DEVICE).bfloat16() for _ in range(3))
    rate = 0.1 * torch.rand(64, device=DEVICE)
    gz, gx, rows = torch.empty_like(z), torch.empty_like(z), torch.empty(65536 * 64, device=DEVICE)

    def seconds(call):
        times = []
        for _ in range(4):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                call()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    scan = seconds(lambda: ops._load_extension().fullscan_backward_softplus(z, rate, out, go, gz,
                                                                            gx, rows))
    assert seconds(lambda: fpscan_amd.scan_backward_softplus(z, rate, out, go)) < 2 * scan


def test_empty_batch_has_zero_rate_gradient():
    z = torch.empty(0, 5, 64, device=DEVICE)
    gz, gr, gx = fpscan_amd.scan_backward_softplus(z, torch.rand(5, device=DEVICE), z, z)
    assert gz.shape == gx.shape == z.shape and (gr == 0).all() and gr.shape == (5,)
