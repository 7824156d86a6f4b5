"""Names of the device kernels that a call runs, as the tracer of torch.profiler sees them (the library's own profile records
name the main launches only)."""
import re

import torch
from torch.profiler import ProfilerActivity, profile


def kernels(call):
    """["gms_rows_kernel", ...]: this library's kernels among those that `call` queues, by their function names, in order."""
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    device = sorted((e for e in p.events() if e.device_type == torch.autograd.DeviceType.CUDA and "fgms::" in e.name), key=lambda e: e.time_range.start)
    return [re.search(r"(\w+)(<|\()", e.name.replace("(anonymous namespace)::", "").split("fgms::", 1)[1]).group(1) for e in device]
