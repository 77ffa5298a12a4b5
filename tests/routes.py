"""The GPU kernels that a call launches, by name."""
import re


def kernels(fn):
    """The set of kernel names (without namespaces and arguments) that fn() launches."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return {m.group(1) for e in prof.events() if (m := re.search(r"(\w+)(<|\()", e.name))
            and "katsu" in e.name}
