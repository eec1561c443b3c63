"""dimwise_forward's row kernel selects with both halves of a wave on chunks of 32 groups: the
winner must be the first strict maximum over all earlier groups, wherever it lies and however
many candidates tie. Integer data, bit for bit against the oracle."""
import pytest
import torch

import fpscan_amd
import oracle
from fpscan_amd import ops
from scan_helpers import DEVICE, DTYPES, bits_equal

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device (MI355X)"),
]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("seqlen", [1024, 2048, 4096, 8192])  # 16 groups, then 32
def test_first_strict_maximum(dtype, seqlen):
    D, G = 40, fpscan_amd.dimwise_groups(seqlen)
    W = oracle.DIMWISE_GEOMETRY[seqlen][0]
    P = oracle.DIMWISE_GEOMETRY[seqlen][1]
    ax = torch.zeros(1, D, seqlen)
    # gates 0 and one nonzero token per group, at its end: v[g] = that token, in {1, 2}
    bx = torch.zeros(1, D, seqlen)
    gen = torch.Generator().manual_seed(seqlen)
    bx[..., P - 1::P] = torch.randint(1, 3, (1, D, seqlen // P), generator=gen).float()
    # keys: few values, many ties; each row's maximum at its own place, in both halves
    bh = torch.randint(-2, 1, (1, D, G), generator=gen).float()
    for d in range(D):
        bh[0, d, d % W] = 1.0
        if d % 3 == 0:
            bh[0, d, (d + 16) % W] = 1.0  # a tie across the halves
    w = torch.zeros(D)
    args = [t.to(dtype) for t in (ax, bx, bh, w, w)]
    want = torch.from_numpy(oracle.dimwise_f64(*args))
    assert want.abs().max() < 256
    ops.set_tiling(1)
    try:
        dev = [t.to(DEVICE) for t in args]
        fpscan_amd.dimwise_forward(*dev)
    finally:
        ops.set_tiling(0)
    assert bits_equal(dev[1].cpu(), want.to(dtype))
