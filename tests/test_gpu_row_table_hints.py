"""Sort layers that the tables per weight row serve: the tables per batch row are left out once three calls have not needed them, and
are there again soon after the layer's operands change to such as do.  The same bits throughout; kernels counted from those that ran."""
import pytest
import torch

pytestmark = pytest.mark.gpu
Q, K = 0.75, 10


def _row_tables(fn, calls):
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        for _ in range(calls):
            fn()
            torch.cuda.synchronize()
    return sum("rc_tables_kernel" in e.name for e in prof.events())


@pytest.mark.parametrize("form", ["values", "interval", "positions"])
def test_tables_per_batch_row_come_and_go(form):
    from sortnet_amd import _lib, ext
    B, N, M = 300, 1056, 1030
    g = torch.Generator().manual_seed(5)
    x, w = torch.empty(B, N, 1, device="cuda"), torch.empty(M, N, device="cuda")
    o = [torch.full((B, M, 1), 7.0, device="cuda") for _ in range(2)] + [torch.full((K, B, M, 1), 7, device="cuda", dtype=torch.int32)]

    def call():
        if form == "values":
            ext.sort_neuron_forward_nograd(x, w, o[0], 1, Q, K)
        elif form == "positions":
            ext.sort_neuron_forward(x, w, o[0], o[2], 1, Q, K)
        else:
            ext.bound_sort_neuron_forward(x - 0.02, x + 0.02, w, o[0], o[1], 1, Q, K)

    def every_term():
        _lib.set_sort_candidate_density(0.0)
        call()
        _lib.set_sort_candidate_density(-1.0)
        return [t.clone() for t in o]

    def same(want):
        call()
        assert all(torch.equal(a, b) for a, b in zip(o, want))

    x.copy_(torch.randn(B, N, 1, generator=g) * 0.05)
    w.copy_(torch.randn(M, N, generator=g))
    alike = every_term()
    for _ in range(4):
        same(alike)
        torch.cuda.synchronize()
    assert _row_tables(call, 12) == 0
    same(alike)
    x.copy_(torch.rand(B, N, 1, generator=g))
    w.copy_(torch.randn(M, N, generator=g) * N ** -0.5)
    images = every_term()
    for _ in range(3):
        same(images)
        torch.cuda.synchronize()
    assert _row_tables(call, 8) >= 7
    same(images)
    assert _lib.last_forward_term_share() < 1.0


@pytest.mark.parametrize("form", ["values", "interval", "positions"])
@pytest.mark.parametrize("every", [2, 7])
def test_operands_that_alternate(form, every):
    """One layer whose operands are served by the tables per weight row in all calls but each `every`-th, which those per batch row serve: after
    a few rounds no call forms every term any more."""
    from sortnet_amd import _lib, ext
    B, N, M = 512, 1056, 1030
    g = torch.Generator().manual_seed(5)
    w = torch.randn(M, N, generator=g).cuda() * N ** -0.5
    alike, images = (torch.randn(B, N, 1, generator=g) * 0.05 * N ** -0.5).cuda(), torch.rand(B, N, 1, generator=g).cuda()
    o, pos = [torch.empty(B, M, 1, device="cuda") for _ in range(2)], torch.empty(K, B, M, 1, device="cuda", dtype=torch.int32)

    def share(x):
        if form == "values":
            ext.sort_neuron_forward_nograd(x, w, o[0], 1, Q, K)
        elif form == "positions":
            ext.sort_neuron_forward(x, w, o[0], pos, 1, Q, K)
        else:
            ext.bound_sort_neuron_forward(x - 1e-4, x + 1e-4, w, o[0], o[1], 1, Q, K)
        return _lib.last_forward_term_share()   # (waits for the stream)

    for _ in range(6):
        assert share(alike) < 1.0
    shares = [share(images if k % every == 0 else alike) for k in range(6 * every)]
    assert max(shares[4 * every:]) < 1.0, shares
