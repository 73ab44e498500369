"""Which kernels a call launches."""

import torch


def launched(call):
    """Names of the kernels that a call launches."""
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    return [e.name for e in p.events() if e.device_type == torch.autograd.DeviceType.CUDA]
