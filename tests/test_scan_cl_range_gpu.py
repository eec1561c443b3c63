"""Channel-last blocks where values leave fp32's range: gates whose product over a tile overflows
while the states stay finite, products that underflow under a state of Inf, and states that
overflow. Every value is what the serial recurrence gives, step after step in fp32, and a column
with such values leaves its neighbours as they are without it.
"""
import pytest
import torch

import fpscan_amd
from scan_helpers import DEVICE, DTYPES, NORM_TOL, bits_equal

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device (MI355X)"),
]

# (batch, seqlen, 16-byte vectors per row): on the 128-byte lines, one tile and 11, few chains and 48
# (the backward's two tile lengths); off the lines, rows of 1 vector (tiles of 512 steps) and 9
SHAPES = [(1, 250, 8), (2, 2600, 8), (2, 1100, 24 * 8), (2, 6000, 1), (1, 2600, 9)]


def serial(a, x, reverse):
    """The recurrence in fp32, one step after the other along axis 1."""
    a, x = a.float(), x.float()
    y = torch.empty_like(x)
    steps = range(x.shape[1])
    last = None
    for t in (reversed(steps) if reverse else steps):
        last = x[:, t] if last is None else a[:, t] * last + x[:, t]
        y[:, t] = last
    return y


def same(got, want, dtype, what):
    got, want = got.cpu().float(), want.to(dtype).float()
    assert torch.equal(torch.isnan(got), torch.isnan(want)), f"{what}: NaN elsewhere"
    inf = torch.isinf(want)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], want[inf]), f"{what}: Inf"
    ok = torch.isfinite(want)
    got, want = torch.where(ok, got, 0).double(), torch.where(ok, want, 0).double()
    # column by column, each over its own size
    err = (got - want).norm(dim=1) / want.norm(dim=1).clamp(min=1e-30)
    assert err.max() <= NORM_TOL[dtype], f"{what}: {err.max():.3e}"


def inputs(kind, shape, dtype):
    """Gates and tokens in processing order; odd columns ordinary, even ones special."""
    B, L, nv = shape
    D = nv * (16 // torch.empty((), dtype=dtype).element_size())
    gen = torch.Generator().manual_seed(L + D)
    a = 0.9 + 0.09 * torch.rand(B, L, D, generator=gen)
    x = torch.randn(B, L, D, generator=gen)
    plain = a.to(dtype), x.to(dtype)
    a, x = a.clone(), x.clone()
    even = slice(0, None, 2)
    grow = L * 3 // 5
    if kind == "growing":  # the product overflows (1.5 ** 219 and more), the state is 0 until late
        a[:, :grow, even] = 1.5
        x[:, :grow - 4, even] = 0.0
    elif kind == "inf_state":  # Inf early on, then products that underflow
        a[:, :, even] = 0.25
        x[:, L // 20, even] = float("inf")
    elif kind == "inf_tiny":  # they underflow within a lane's steps
        a[:, :, even] = 1e-6
        x[:, L // 20, even] = float("inf")
    elif kind == "nan_state":
        x[:, L // 20, even] = float("nan")
    else:  # "overflow": the state itself overflows
        a[:, :, even] = 1.5
        x[:, :, even] = 1.0
    return plain, (a.to(dtype), x.to(dtype))


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("kind", ["growing", "inf_state", "inf_tiny", "nan_state", "overflow"])
def test_as_the_serial_recurrence(kind, shape, dtype):
    plain, special = inputs(kind, shape, dtype)
    overruns = fpscan_amd.lookback_overruns()
    for reverse in (False, True):
        turn = (lambda t: t.flip(1)) if reverse else (lambda t: t)
        run = lambda p: fpscan_amd.scan_forward_channel_last(  # noqa: E731
            *(turn(t).to(DEVICE) for t in p), reverse)
        y = run(special)
        same(y, serial(*(turn(t) for t in special), reverse), dtype, f"reverse={reverse}")
        assert bits_equal(y[..., 1::2], run(plain)[..., 1::2]), "ordinary columns"

    # the backward, reversed in time: grad_tokens[t] = grad_out[t] + gates[t + 1] grad_tokens[t + 1]
    def backward(p):
        a, go = (t.flip(1) for t in p)
        out = torch.ones_like(go)
        gates = torch.cat([torch.ones_like(a[:, :1]), a[:, :-1]], 1)
        return a, fpscan_amd.scan_backward_channel_last(*(t.to(DEVICE) for t in (gates, out, go)))

    a, (gg, gx) = backward(special)
    want = serial(a, special[1].flip(1), True)
    same(gx, want, dtype, "grad_tokens")
    same(gg[:, 1:], want[:, 1:], dtype, "grad_gates with out = 1")
    # before the first step out is 0
    first = want[:, 0].to(dtype).float() * 0.0
    assert torch.equal(torch.isnan(gg[:, 0].cpu()), torch.isnan(first))
    ordinary = backward(plain)[1]
    assert bits_equal(gg[..., 1::2], ordinary[0][..., 1::2])
    assert bits_equal(gx[..., 1::2], ordinary[1][..., 1::2])
    assert fpscan_amd.lookback_overruns() == overruns
