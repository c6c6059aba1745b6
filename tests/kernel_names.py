"""Which kernels a call launches, by the names that torch's profiler records for
the process: a test of a kernel says with it that the kernel ran."""
import re


def kernels_of(call):
    """Names of the library's kernels that call() launches, template arguments
    with them, e.g. "decode_route_kernel<4>"."""
    import warnings

    from torch.profiler import ProfilerActivity, profile

    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        with profile(activities=[ProfilerActivity.CUDA]) as p:
            call()
    names = [re.search(r"moe::(?:\(anonymous namespace\)::)?(\w+(?:<[^>]*>)?)\(", e.key) for e in p.key_averages()]
    return {m.group(1) for m in names if m}
