"""GPU tests of the block channel-last scan, which the automatic choice takes where one pass per
strip lacks strips: one tile of 256 threads per workgroup, panels of up to 8 (rows off the
128-byte lines: up to 32) 16-byte vectors, 4 or 8 steps per lane, a look-back of depth 8.

Against the oracle on integer data bit for bit (gates 0 or 1, every partial result exact) and
on random data, at the edges of tiles, panels and look-back depth; its workspace bounds,
padded strides, in-place use, determinism, and a look-back wait that gives up.
"""
import pytest
import torch

import fpscan_amd
import oracle
from fpscan_amd import ops
from scan_helpers import DEVICE, DTYPES, bits_equal, check
from test_scan_cl_tiled_gpu import _CODE, cl_inputs, lib  # noqa: F401  (fixture)

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device (MI355X)"),
]

# (batch, seqlen, 16-byte vectors per row): on the lines, 8 vectors = 32 groups: tiles of 256
# steps (8 per lane), of 128 in the backward from 48 chains; one tile exactly, one step less
# and more; 11 tiles (an end value two look-backs back); off the lines, whole rows as panels
# (1, 2, 9, 31 vectors: 64, 64, 28, 8 groups) and split ones (33 -> 5 panels of 7); 2 batches of
# 24 panels: the backward's shorter tiles
SHAPES = [(1, 255, 8), (2, 256, 8), (1, 257, 8), (1, 2600, 8), (3, 300, 16), (2, 2049, 1),
          (1, 4500, 2), (2, 3000, 9), (3, 700, 31), (1, 1000, 33), (2, 1300, 24 * 8), (5, 1, 40),
          (2, 127, 24 * 8), (2, 129, 24 * 8)]


def _shape(shape, dtype):
    B, L, nv = shape
    return B, L, nv * (16 // torch.empty((), dtype=dtype).element_size())


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_exact_on_integer_data(dtype, shape):
    shape = _shape(shape, dtype)
    gen = torch.Generator().manual_seed(sum(shape))
    g = (torch.randint(0, 6, shape, generator=gen) > 0).to(dtype)
    x = torch.randint(-2, 3, shape, generator=gen).to(dtype)
    go = torch.randint(-2, 3, shape, generator=gen).to(dtype)
    gd, xd, god = g.to(DEVICE), x.to(DEVICE), go.to(DEVICE)
    ext = ops._load_extension()
    for rev in (False, True):
        want = torch.from_numpy(oracle.scan_f64_channel_last(g, x, rev))
        assert want.abs().max() < 256  # exact in every dtype
        assert bits_equal(fpscan_amd.scan_forward_channel_last(gd, xd, rev).cpu(), want.to(dtype))
        y = xd.clone()
        fpscan_amd.scan_forward_channel_last(gd, y, rev, out=y)
        assert bits_equal(y.cpu(), want.to(dtype)), "in place"
    want = torch.from_numpy(oracle.scan_f64_channel_last(g, x, False)).to(dtype)
    out = torch.full_like(xd, float("nan"))
    ext.fullscan_forward_cl_saved(gd, xd, out)
    assert bits_equal(out.cpu(), want), "the forward of a training step"
    gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(g, want, go)
    assert abs(gx_ref).max() < 256 and (dtype != torch.bfloat16 or abs(gg_ref).max() < 2 ** 16)
    gg, gx = fpscan_amd.scan_backward_channel_last(gd, out, god)
    assert bits_equal(gx.cpu(), torch.from_numpy(gx_ref).to(dtype))
    # one rounding of an exact fp32 product
    assert bits_equal(gg.cpu(), torch.from_numpy(gg_ref).to(dtype))


# off the lines, rows of 17 to 32 vectors: whole (from 4 sequences in the backward, 64 in the
# forward, up to 20 vectors from 4 in both) and split
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", [(1, 1500, 15), (1, 1500, 17), (3, 700, 31), (4, 700, 31),
                                   (3, 500, 20 - 1), (4, 500, 20), (4, 500, 21), (63, 150, 29),
                                   (64, 150, 29)], ids=str)
def test_whole_and_split_rows(dtype, shape):
    test_exact_on_integer_data(dtype, shape)


# off the lines with 512 strips or more: blocks up to 16 vectors (2 tiles and 1), up to 32 from 256
# steps, the one pass otherwise
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", [(513, 130, 15), (512, 120, 15), (512, 255, 17), (512, 256, 17),
                                   (512, 65, 31), (256, 257, 65)], ids=str)
def test_enough_strips_off_the_lines(dtype, shape):
    test_short_sequences(dtype, shape)


# around the length from which a sequence within one tile takes a block: 32 steps (the backward 16),
# more with many chains, 96 at most; chains of 8 vectors on the lines, of up to 8 off them
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", [(1, 15, 8), (1, 16, 8), (1, 31, 8), (1, 32, 8), (2, 31, 33),
                                   (2, 32, 33), (16, 51, 8 * 64), (16, 52, 8 * 64),
                                   (30, 95, 8 * 64), (30, 96, 8 * 64)], ids=str)
def test_short_sequences(dtype, shape):
    shape = _shape(shape, dtype)
    g, x = cl_inputs(*shape, dtype, seed=3)
    go = torch.randn(shape, generator=torch.Generator().manual_seed(5)).to(dtype)
    y = fpscan_amd.scan_forward_channel_last(g.to(DEVICE), x.to(DEVICE))
    check(y, oracle.scan_f64_channel_last(g, x), dtype, "forward")
    gg, gx = fpscan_amd.scan_backward_channel_last(g.to(DEVICE), y, go.to(DEVICE))
    gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(g, y.cpu(), go)
    check(gx, gx_ref, dtype, "grad_tokens")
    check(gg, gg_ref, dtype, "grad_gates")


@pytest.mark.parametrize("shape", [(62, 5, 3248), (24, 1, 5856), (134, 8, 1280)], ids=str)
def test_a_few_steps_cost_no_more_than_the_one_pass(shape):
    g, x, go = (torch.rand(shape, device=DEVICE).bfloat16() for _ in range(3))
    out, gg, gx = (torch.empty_like(x) for _ in range(3))
    ext = ops._load_extension()

    def microseconds(call):
        times = []  # the smallest of them: the host limits some
        for _ in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(50):
                call()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 20)
        return min(times)

    for call in (lambda: ext.fullscan_forward_cl(g, x, out, False),
                 lambda: ext.fullscan_backward_cl(g, out, go, gg, gx)):
        automatic = microseconds(call)
        ops.set_tiling(1)
        try:
            one_pass = microseconds(call)
        finally:
            ops.set_tiling(0)
        assert automatic < 2 * one_pass


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shape", [(1, 20000, 8), (2, 5000, 33), (4, 2500, 96)], ids=str)
def test_matches_oracle_is_deterministic_and_mirrored(dtype, shape):
    g, x = cl_inputs(*_shape(shape, dtype), dtype, seed=7)
    go = torch.randn(g.shape, generator=torch.Generator().manual_seed(5)).to(dtype)
    gd, xd = g.to(DEVICE), x.to(DEVICE)
    y = fpscan_amd.scan_forward_channel_last(gd, xd)
    check(y, oracle.scan_f64_channel_last(g, x), dtype, f"blocks {shape}")
    for _ in range(3):
        assert bits_equal(fpscan_amd.scan_forward_channel_last(gd, xd), y)
    mirrored = fpscan_amd.scan_forward_channel_last(gd.flip(1), xd.flip(1), reverse=True).flip(1)
    assert bits_equal(mirrored, y)
    gg, gx = fpscan_amd.scan_backward_channel_last(gd, y, go.to(DEVICE))
    gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(g, y.cpu(), go)
    check(gx, gx_ref, dtype, "grad_tokens")
    check(gg, gg_ref, dtype, "grad_gates")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("nv,pad", [(8, 8), (9, 4), (40, 3)], ids=str)
def test_padded_strides_and_workspace_bounds(lib, dtype, nv, pad):  # noqa: F811
    """Rows inside a wider buffer, on and off the lines, with the workspace between guards."""
    B, L, D = _shape((2, 2700, nv), dtype)
    vec = D // nv
    st, code = D + pad * vec, _CODE[dtype]
    sb = L * st
    g, x = cl_inputs(B, L, D, dtype, seed=4)
    go = torch.randn(B, L, D, generator=torch.Generator().manual_seed(2)).to(dtype)

    def embed(t):
        buf = torch.full((B, L, st), -3.0, dtype=dtype, device=DEVICE)
        buf[:, :, :D] = t.to(DEVICE)
        return buf

    def ws(op):
        n = lib.fpscan_workspace_bytes_cl(B, L, D, st, code, op)
        buf = torch.full((n + 512,), 0xA5, dtype=torch.uint8, device=DEVICE)
        return buf, buf.data_ptr() + 256, n

    gb, xb, gob = embed(g), embed(x), embed(go)
    outb, ggb, gxb = (embed(torch.zeros_like(x)) for _ in range(3))
    stream = torch.cuda.current_stream().cuda_stream
    w0, p0, n0 = ws(0)
    w1, p1, n1 = ws(1)
    assert lib.fpscan_scan_fwd_cl(gb.data_ptr(), xb.data_ptr(), outb.data_ptr(), B, L, D, sb, st,
                                  code, 0, p0, n0, stream) == 0
    assert lib.fpscan_scan_bwd_cl(gb.data_ptr(), outb.data_ptr(), gob.data_ptr(), ggb.data_ptr(),
                                  gxb.data_ptr(), B, L, D, sb, st, code, p1, n1, stream) == 0
    torch.cuda.synchronize()
    for w, n in ((w0, n0), (w1, n1)):
        assert (w[:256] == 0xA5).all() and (w[256 + n:] == 0xA5).all(), "workspace overrun"
    out = outb[:, :, :D].cpu()
    check(out, oracle.scan_f64_channel_last(g, x), dtype, "strided fwd")
    gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(g, out, go)
    check(gxb[:, :, :D].cpu(), gx_ref, dtype, "strided grad_tokens")
    check(ggb[:, :, :D].cpu(), gg_ref, dtype, "strided grad_gates")
    for buf in (outb, ggb, gxb):
        assert (buf[:, :, D:] == -3.0).all(), "padding was written"


@pytest.mark.parametrize("op", ["fwd", "rev", "bwd"])
def test_overrun_poisons_and_is_counted(op):
    """One chain of 12 tiles of 256 steps; tile 1 never publishes, so tiles 2..9, which compose
    its aggregate, are NaN, tiles 0 and 1 are right, and no value is anything else."""
    L, steps = 12 * 256, 256
    gen = torch.Generator().manual_seed(3)
    g = (0.9 + 0.1 * torch.rand(1, L, 32, generator=gen)).to(DEVICE)
    x, go = (torch.randn(1, L, 32, generator=gen).to(DEVICE) for _ in range(2))
    y = fpscan_amd.scan_forward_channel_last(g, x)

    def run():
        if op == "bwd":
            return list(fpscan_amd.scan_backward_channel_last(g, y, go))
        return [fpscan_amd.scan_forward_channel_last(g, x, op == "rev")]

    want, before = run(), fpscan_amd.lookback_overruns()
    ops.set_lookback_test_hook(1, 64)
    try:
        got = run()
        torch.cuda.synchronize()
    finally:
        ops.set_lookback_test_hook()
    assert fpscan_amd.lookback_overruns() > before
    for a, b in zip(got, want):
        if op != "fwd":
            a, b = a.flip(1), b.flip(1)
        assert bits_equal(a[:, :2 * steps], b[:, :2 * steps])
        assert torch.isnan(a[:, 2 * steps:10 * steps]).all()
        nan = torch.isnan(a)
        assert bits_equal(a[~nan], b[~nan])


# rows of 1 to 3 vectors: one tile of up to 2048 steps; several of 512 steps while all are resident
# (1024 workgroups in the forward, 768 in the backward) and a chain has at most 32; longer ones otherwise
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape,vectors", [((4, 2048), 1), ((4, 2049), 1), ((2, 16384), 1),
                                           ((2, 16385), 1), ((3, 1025), 2), ((3, 681), 3),
                                           ((204, 2049), 1), ((154, 2049), 1), ((205, 2049), 1)],
                         ids=str)
def test_narrow_rows(shape, vectors, dtype):
    test_short_sequences(dtype, (*shape, vectors))


@pytest.mark.parametrize("seqlen,steps", [(2049, 512), (16384, 512), (16385, 1024)])
def test_narrow_rows_take_short_tiles(seqlen, steps):
    """Tile 1 never publishes: the first value that its silence makes NaN is tile 2's."""
    g, x = (torch.rand(1, seqlen, 4, device=DEVICE) for _ in range(2))
    ops.set_lookback_test_hook(1, 64)
    try:
        y = fpscan_amd.scan_forward_channel_last(g, x)
        torch.cuda.synchronize()
    finally:
        ops.set_lookback_test_hook()
    assert torch.isnan(y[0, :, 0]).nonzero()[0].item() == 2 * steps


# the sizes from which the ring of tiles takes over: split rows on 64-byte lines below and from 192
# MiB, the 2-byte backward with 17 chains below and from 512 MiB (16 chains never), against the oracle
# on the first and last columns
@pytest.mark.parametrize("dtype,shape", [
    (torch.float32, (1, 43689, 1152 - 16)), (torch.float32, (1, 44400, 1152 - 16)),
    (torch.bfloat16, (17, 246723, 64)), (torch.bfloat16, (17, 246724, 64)),
    (torch.bfloat16, (16, 262144, 64))], ids=str)
def test_around_the_sizes_of_the_tiles(dtype, shape):
    gen = torch.Generator(device=DEVICE).manual_seed(shape[1])
    g = (0.99 + 0.01 * torch.rand(shape, generator=gen, device=DEVICE)).to(dtype)
    x, go = (torch.randn(shape, generator=gen, device=DEVICE).to(dtype) for _ in range(2))
    y = fpscan_amd.scan_forward_channel_last(g, x)
    gg, gx = fpscan_amd.scan_backward_channel_last(g, y, go)
    at = [t[:1, :, [0, -1]].cpu() if b == 0 else t[-1:, :, [0, -1]].cpu()
          for b in (0, 1) for t in (g, x, go, y, gg, gx)]
    for g1, x1, go1, y1, gg1, gx1 in (at[:6], at[6:]):
        check(y1, oracle.scan_f64_channel_last(g1, x1), dtype, "forward")
        gg_ref, gx_ref = oracle.scan_bwd_f64_channel_last(g1, y1, go1)
        check(gx1, gx_ref, dtype, "grad_tokens")
        check(gg1, gg_ref, dtype, "grad_gates")
    assert torch.isfinite(y).all() and torch.isfinite(gg).all() and torch.isfinite(gx).all()
