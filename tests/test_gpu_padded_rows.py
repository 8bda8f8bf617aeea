"""Sort neuron of layers whose rows are no multiple of 32 inputs, on padded copies: one to 31 inputs missing, one batch row, batch
tiles that are not full, tables that serve and tables that do not, ties, undefined inputs; a stream under capture that has not run
the call.  Values, bounds and positions bit for bit against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
Q, K = 0.75, 10


def _data(B, N, M, spread, seed=0):
    g = torch.Generator().manual_seed(B + N + seed)
    return torch.randn(B, N, 1, generator=g) * spread, torch.randn(M, N, generator=g)


def _run(x, w):
    from sortnet_amd import ext
    B, M = x.shape[0], w.shape[0]
    new = lambda *s: torch.full(s, 7.0, device="cuda")   # noqa: E731
    y, yp, lo, up, pos = new(B, M, 1), new(B, M, 1), new(B, M, 1), new(B, M, 1), torch.full((K, B, M, 1), 7, device="cuda", dtype=torch.int32)
    ext.sort_neuron_forward_nograd(x, w, y, 1, Q, K)
    ext.sort_neuron_forward(x, w, yp, pos, 1, Q, K)
    ext.bound_sort_neuron_forward(x - 0.03, x + 0.03, w, lo, up, 1, Q, K)
    return y, yp, pos, lo, up


@pytest.mark.parametrize("B,N,M,spread,kind", [
    (1, 4129, 4100, 0.3, ""), (129, 1055, 140, 0.05, "odd"), (70, 1567, 161, 0.3, "ties"), (300, 335, 300, 3.0, ""), (260, 1030, 130, 0.3, "odd"),
    (64, 4081, 65, 1.0, "ties"), (33, 2049, 251, 0.05, ""), (130, 12290, 11, 0.3, "")])
def test_against_the_oracle(oracle, B, N, M, spread, kind):
    x, w = _data(B, N, M, spread)
    if kind == "ties":
        x, w = (x * 4).round() / 4, (w * 4).round() / 4
    if kind == "odd":
        x[0, 3], w[1, 2], x[1, N - 1], w[2, N - 1] = float("nan"), float("inf"), float("inf"), float("nan")
    y, yp, pos, lo, up = _run(x.cuda(), w.cuda())
    ry, rp = oracle.sort_neuron_forward(x.numpy(), w.numpy(), Q, K)
    rl, ru = oracle.bound_sort_neuron_forward((x - 0.03).numpy(), (x + 0.03).numpy(), w.numpy(), Q, K)
    for got, want in ((y, ry), (yp, ry), (lo, rl), (up, ru)):
        np.testing.assert_array_equal(got.cpu().numpy(), want)
    np.testing.assert_array_equal(pos.cpu().numpy(), np.asarray(rp).astype(np.int32).reshape(tuple(pos.shape)))


def test_tables_serve_and_capture_needs_no_scratch():
    from sortnet_amd import _lib
    x, w = (t.cuda() for t in _data(128, 1306, 1306, 0.05))
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        fresh = _run(x, w)                       # a stream without a workspace: every term
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        want = _run(x, w)
        assert _lib.last_forward_term_share() < 0.5
        for a, b in zip(fresh, want):
            assert torch.equal(a, b)
            a.zero_()


@pytest.mark.parametrize("B,N,M,kind", [(129, 1057, 1030, ""), (64, 4081, 530, "ties"), (33, 5121, 840, "odd"), (257, 2050, 4130, ""),
                                        (70, 5829, 5270, "odd"), (131, 9998, 1645, "ties")])
def test_interval_bounds_against_the_oracle(oracle, B, N, M, kind):
    from sortnet_amd import ext
    x, w = _data(B, N, M, 0.5)
    w *= N ** -0.5
    if kind == "ties":
        x, w = (x * 8).round() / 8, (w * 64).round() / 64
    lo, up = x - 0.03, x + 0.03
    if kind == "odd":
        lo[0, 3], w[1, 2], up[1, N - 1], w[2, N - 1], lo[2, 5] = float("nan"), float("inf"), float("inf"), float("nan"), up[2, 5] + 1
    # an output depends on its own rows alone: some of the largest layers
    rows, cols = slice(0, B, 1 + B * M * N // 2 ** 28), slice(0, M, 1 + B * M * N // 2 ** 29)
    rl, ru, rpl, rpu = oracle.bound_inf_dist_forward(lo[rows].contiguous().numpy(), up[rows].contiguous().numpy(), w[cols].contiguous().numpy())
    new = lambda t: torch.full((B, M, 1), 7, device="cuda", dtype=t)   # noqa: E731
    l, u, l2, u2, pl, pu = (new(t) for t in (torch.float32,) * 4 + (torch.int32,) * 2)
    ext.bound_inf_dist_forward_nograd(lo.cuda(), up.cuda(), w.cuda(), l, u, 1)
    ext.bound_inf_dist_forward(lo.cuda(), up.cuda(), w.cuda(), l2, u2, pl, pu, 1)
    for got, want in ((l, rl), (u, ru), (l2, rl), (u2, ru), (pl, rpl), (pu, rpu)):
        got = got[rows][:, cols].cpu().numpy()
        np.testing.assert_array_equal(got, np.asarray(want).reshape(got.shape).astype(got.dtype))


@pytest.mark.parametrize("B,N,M,spread", [(99, 2304, 59, 0.3), (16, 320, 250, 0.05), (64, 511, 65, 3.0), (1, 1200, 900, 0.3), (129, 5120, 3, 0.3)])
def test_positions_of_few_outputs(oracle, B, N, M, spread):
    x, w = _data(B, N, M, spread)
    _, yp, pos, _, _ = _run(x.cuda(), w.cuda())
    ry, rp = oracle.sort_neuron_forward(x.numpy(), w.numpy(), Q, K)
    np.testing.assert_array_equal(yp.cpu().numpy(), ry)
    np.testing.assert_array_equal(pos.cpu().numpy(), np.asarray(rp).astype(np.int32).reshape(tuple(pos.shape)))


@pytest.mark.parametrize("B,N,M,q", [(91, 799, 1920, 0.3), (250, 1025, 530, 0.7), (33, 2303, 2001, 0.05), (129, 4097, 261, 1.0), (200, 5131, 140, 0.3)])
def test_factored_mask_against_the_oracle(oracle, B, N, M, q):
    from sortnet_amd import _lib, ext
    x, w = _data(B, N, M, 0.3)
    x[0, N - 1], w[1, 2], w[2, N - 1] = float("nan"), float("inf"), -9.0
    y, y2, pos = (torch.full((B, M, 1), 7, device="cuda", dtype=t) for t in (torch.float32, torch.float32, torch.int32))
    ry, rp = oracle.masked_inf_dist_forward(x.numpy(), w.numpy(), q, 11, oracle.MASK_FACTORED)
    ext.masked_inf_dist_forward(x.cuda(), w.cuda(), y, pos, 1, q, 11, ext.MASK_FACTORED)
    ext.masked_inf_dist_forward(x.cuda(), w.cuda(), y2, None, 1, q, 11, ext.MASK_FACTORED)
    assert _lib.last_forward_kernel().startswith("fwd_kernel_pipe")
    for got, want in ((y, ry), (y2, ry), (pos, rp)):
        np.testing.assert_array_equal(got.cpu().numpy(), np.asarray(want).reshape(B, M, 1).astype(got.cpu().numpy().dtype))


@pytest.mark.parametrize("B,N,M,q,density", [(200, 5131, 140, 0.3, 1.0), (129, 2049, 517, 0.6, 1.0), (257, 4097, 2100, 0.3, None)])
def test_factored_mask_from_tables(oracle, B, N, M, q, density):
    """Padded copies, keep bits of the raw length and candidate tables together: at a forced density, and at the built-in limit (2^31 terms)."""
    from sortnet_amd import _lib, ext
    g = torch.Generator().manual_seed(B)
    x, w = torch.randn(B, N, 1, generator=g) * 0.02, torch.randn(M, N, generator=g)   # (batch rows alike: tables per weight row)
    x[0, N - 1], w[1, 2], w[2, N - 1], w[3] = float("nan"), float("inf"), -9.0, 0.0
    rows, cols = min(B, 40), min(M, 300)   # (a row's keep bits come from its number)
    ry, rp = oracle.masked_inf_dist_forward(x[:rows].numpy(), w[:cols].numpy(), q, 11, oracle.MASK_FACTORED)
    xd, wd = x.cuda(), w.cuda()
    new = lambda t: torch.full((B, M, 1), 7, device="cuda", dtype=t)   # noqa: E731

    def run():
        y, y2, pos = new(torch.float32), new(torch.float32), new(torch.int32)
        ext.masked_inf_dist_forward(xd, wd, y, pos, 1, q, 11, ext.MASK_FACTORED)
        share = _lib.last_forward_term_share()
        ext.masked_inf_dist_forward(xd, wd, y2, None, 1, q, 11, ext.MASK_FACTORED)
        return y, y2, pos, max(share, _lib.last_forward_term_share())

    try:
        _lib.set_linf_candidate_density(0.0)
        *every, share = run()
        assert share == 1.0
        _lib.set_linf_candidate_density(-1.0 if density is None else density)
        *got, share = run()
    finally:
        _lib.set_linf_candidate_density(-1.0)
    assert share < 1.0
    for a, b in zip(got, every):
        assert torch.equal(a, b)
    for a, want in zip(got, (ry, ry, rp)):
        a = a[:rows, :cols].cpu().numpy()
        np.testing.assert_array_equal(a, np.asarray(want).reshape(a.shape).astype(a.dtype))
