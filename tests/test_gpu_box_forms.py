"""Values and bounds of a layer in one call: which sizes share a table."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(B, N, M, width=0.02):
    g = torch.Generator(device="cuda").manual_seed(B + N)
    x = torch.randn(B, N, 1, device="cuda", generator=g) * 0.05
    w = torch.randn(M, N, device="cuda", generator=g)
    return x, x - width, x + width, w, torch.randn(M, device="cuda", generator=g)


def _names(fn):
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events()]


@pytest.mark.parametrize("B,N,M", [(16, 4443, 2400), (10, 4443, 3900), (128, 1306, 500)])
def test_ragged_rows_share_a_table(B, N, M):
    """Rows that are loaded value by value, sizes at which neither the values nor the bounds stream the weights."""
    from sortnet_amd import functional as F
    x, lo, up, w, shift = _operands(B, N, M)
    want = [F._shifted_values(x, w, 1, 0.75, shift, -1.0), *F._shifted_bounds(lo, up, w, 1, 0.75, shift, -1.0)]
    torch.cuda.synchronize()
    got = []
    names = _names(lambda: got.extend(F._shifted_box(x, lo, up, w, 1, 0.75, shift, -1.0)))
    assert any("sc_main_kernel<10, true, false, true>" in n for n in names), names
    assert all(torch.equal(a, b) for a, b in zip(got, want))
