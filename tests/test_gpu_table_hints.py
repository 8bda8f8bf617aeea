"""Layers whose tables do not pay: once three calls have shown it, one call in 32 builds them again, also where the host queues calls
long before the device gets to them and no outcome has come back.  Counted from the kernels that ran."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tables_built(fn, calls, dev):
    from torch.profiler import ProfilerActivity, profile
    a = torch.randn(8192, 8192, device=dev)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        for _ in range(12):
            a = a @ a * 1e-2        # the device is busy while the calls are queued
        for _ in range(calls):
            fn()
        torch.cuda.synchronize()
    names = [e.name for e in prof.events()]
    assert sum("fwd_kernel" in n for n in names) >= calls
    return sum("rc_tables_kernel" in n for n in names)


@pytest.mark.parametrize("positions", [False, True])
def test_a_layer_that_is_queued_ahead_probes_once_in_a_while(positions):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(3)
    B, CI, CO = 400, 1024, 1024
    x = torch.randn(B, CI, 1, generator=g).to(dev)     # everything is marked
    w = torch.randn(CO, CI, generator=g).to(dev)
    xl, xu = x - 0.1, x + 0.1
    o = [torch.empty(B, CO, 1, device=dev) for _ in range(2)]
    p = [torch.empty(B, CO, 1, device=dev, dtype=torch.int32) for _ in range(2)]

    def call():
        if positions:
            ext.bound_inf_dist_forward(xl, xu, w, *o, *p, 1)
        else:
            ext.bound_inf_dist_forward_nograd(xl, xu, w, *o, 1)
    for _ in range(4):
        call()
        torch.cuda.synchronize()
    assert 1 <= _tables_built(call, 100, dev) <= 4      # after 28 to 31 calls, and then after every 31
