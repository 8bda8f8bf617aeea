"""Values and bounds of a layer in one call: which sizes share a table, depths other than the layers' own, and the call without a shift."""
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


@pytest.mark.parametrize("K", [2, 7, 10, 25])
@pytest.mark.parametrize("B,N,M", [(128, 1024, 450), (200, 1306, 700)])
@pytest.mark.parametrize("width", [0.02, 3.0])
def test_depths_and_the_call_without_a_shift(B, N, M, width, K):
    from sortnet_amd import _lib, ext, functional as F
    x, lo, up, w, shift = _operands(B, N, M, width)
    ref = [torch.empty(B, M, 1, device="cuda") for _ in range(3)]
    ext.sort_neuron_forward_nograd(x, w, ref[0], 1, 0.75, K)
    ext.bound_sort_neuron_forward(lo, up, w, ref[1], ref[2], 1, 0.75, K)
    st = torch.cuda.current_stream().cuda_stream
    for _ in range(5):
        out = [torch.empty(B, M, 1, device="cuda") for _ in range(3)]
        _lib.call("sd_sort_neuron_box_forward", *(t.data_ptr() for t in (x, lo, up, w)), B, M, N, 1, 1, *(t.data_ptr() for t in out), 0.75, K,
                  None, 0.0, st)
        assert all(torch.equal(a, b) for a, b in zip(out, ref))
        for a, b in zip(F._shifted_box(x, lo, up, w, 1, 0.75, shift, -1.0, truncate=K), ref):
            assert torch.equal(a, b - shift.view(1, -1, 1))
        torch.cuda.synchronize()
