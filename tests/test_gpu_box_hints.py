"""Layers whose values and bounds come from one table: which other tables are queued beside it.  Counted from the kernels that ran; the same
bits as the two calls by themselves throughout."""
import pytest
import torch

pytestmark = pytest.mark.gpu
Q = 0.75


class _Layer:
    def __init__(self, B, N, M, seed=5):
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.w = torch.randn(M, N, device="cuda", generator=g)
        self.x = torch.randn(B, N, 1, device="cuda", generator=g) * 0.05
        self.shift = torch.randn(M, device="cuda", generator=g)

    def box(self, width):
        from sortnet_amd import functional as F
        return F._shifted_box(self.x, self.x - width, self.x + width, self.w, 1, Q, self.shift, -1.0)

    def apart(self, width):
        from sortnet_amd import functional as F
        return (F._shifted_values(self.x, self.w, 1, Q, self.shift, -1.0),
                *F._shifted_bounds(self.x - width, self.x + width, self.w, 1, Q, self.shift, -1.0))


def _names(fn):
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events()]


def _count(names, part):
    return sum(part in n for n in names)


def test_tables_per_batch_row_are_left_out():
    """Where the shared table serves, those per batch row are left out after three calls, of the values and of the bounds."""
    layer = _Layer(300, 1056, 1030)
    want = layer.apart(0.02)
    for _ in range(4):
        assert all(torch.equal(a, b) for a, b in zip(layer.box(0.02), want))
        torch.cuda.synchronize()

    def twelve():
        for _ in range(12):
            layer.box(0.02)
            torch.cuda.synchronize()
    names = _names(twelve)
    assert _count(names, "sc_main_kernel") >= 12
    assert _count(names, "rc_tables_kernel") == 0, names
    assert all(torch.equal(a, b) for a, b in zip(layer.box(0.02), want))


def test_values_beside_intervals_that_alternate():
    """Narrow and wide intervals in turn, the wide ones beyond the shared table: after a few rounds the values' own tables stand in for it in
    every wide call, and they are left out again where the intervals stay narrow."""
    layer = _Layer(300, 1056, 1030)
    want = {width: layer.apart(width) for width in (0.02, 3.0)}

    def call(width):
        assert all(torch.equal(a, b) for a, b in zip(layer.box(width), want[width]))
        torch.cuda.synchronize()
    own = "sc_main_kernel<10, false"
    for _ in range(5):
        call(0.02)
    assert _count(_names(lambda: call(0.02)), own) == 0
    for _ in range(2):
        call(3.0)
        call(0.02)
    for _ in range(6):
        names = _names(lambda: call(3.0))
        assert _count(names, own) == 1, names
        call(0.02)
    for _ in range(14):
        call(0.02)
    assert _count(_names(lambda: call(0.02)), own) == 0
