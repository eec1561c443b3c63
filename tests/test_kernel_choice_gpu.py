"""Which kernel a call launches, by the name that the profiler records: the rules that give the same
results either way and would otherwise show only in the time.
"""
import re

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

import fpscan_amd
from scan_helpers import DEVICE

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
