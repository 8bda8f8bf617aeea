"""The kernels that stream the weights past few batch rows (a wavefront per weight row), against the oracle: values,
positions and bounds bit for bit, weighted sums at the bar of every sort-neuron test (same products and sums in fp32)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# batch rows, inputs per group, outputs per group, groups: one input, less than a wavefront, one over and under the
# register tiles (1024, 3072, 5120, 10240 inputs), rows that are no multiple of four, more wavefronts than weight rows,
# several slices of the batch rows, groups
SHAPES = [(1, 1, 1, 1), (2, 5, 3, 1), (3, 63, 9, 1), (4, 64, 4, 1), (5, 1024, 7, 1), (2, 1028, 5, 1), (3, 1025, 6, 1),
          (2, 3072, 9, 1), (1, 3076, 8, 1), (2, 5120, 3, 1), (2, 5124, 5, 1), (1, 10240, 2, 1), (2, 10239, 3, 1),
          (17, 200, 33, 1), (6, 130, 10, 3), (70, 96, 5, 2)]
KINDS = ["normal", "ties", "undefined"]


def _data(shape, kind):
    B, n, m, G = shape
    g = torch.Generator().manual_seed(B * 31 + n + m)
    if kind == "ties":
        x = torch.randint(0, 4, (B, n * G, 1), generator=g).float()
        w = torch.randint(0, 4, (m * G, n), generator=g).float()
    else:
        x, w = torch.randn(B, n * G, 1, generator=g), torch.randn(m * G, n, generator=g)
    if kind == "undefined":
        x[torch.rand(x.shape, generator=g) < 0.02] = float("nan")
        w[torch.rand(w.shape, generator=g) < 0.02] = float("nan")
        w[torch.rand(w.shape, generator=g) < 0.01] = float("inf")
    return x, w


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_streamed_layers_match_oracle(oracle, shape, kind):
    from sortnet_amd import _lib, ext
    B, n, m, G = shape
    x, w = _data(shape, kind)
    xd, wd = x.cuda(), w.cuda()
    new = lambda: torch.empty(B, m * G, 1, device="cuda")                     # noqa: E731
    newi = lambda: torch.empty(B, m * G, 1, device="cuda", dtype=torch.int32)  # noqa: E731
    y, y2, p, p2 = new(), new(), newi(), newi()

    def streamed():
        assert _lib.last_forward_kernel().startswith("row_stream_kernel"), _lib.last_forward_kernel()

    def same(got, ref):
        assert np.array_equal(got.cpu().numpy(), np.asarray(ref).reshape(tuple(got.shape)), equal_nan=True)

    ry, rp = oracle.inf_dist_forward(x.numpy(), w.numpy(), groups=G)
    ext.inf_dist_forward_nograd(xd, wd, y, G)
    streamed()
    same(y, ry)
    ext.inf_dist_forward(xd, wd, y, p, G)
    streamed()
    same(y, ry)
    same(p, rp)
    ry, rp = oracle.masked_inf_dist_forward(x.numpy(), w.numpy(), 0.4, 11, oracle.MASK_FACTORED, groups=G)
    ext.masked_inf_dist_forward(xd, wd, y, p, G, 0.4, 11, ext.MASK_FACTORED)
    streamed()
    same(y, ry)
    same(p, rp)
    lo, up = x - 0.1, x + 0.2
    up[:, ::7] = lo[:, ::7] - 0.05                                           # inverted intervals
    rl, ru, rpl, rpu = oracle.bound_inf_dist_forward(lo.numpy(), up.numpy(), w.numpy(), groups=G)
    ext.bound_inf_dist_forward_nograd(lo.cuda(), up.cuda(), wd, y, y2, G)
    streamed()
    same(y, rl)
    same(y2, ru)
    ext.bound_inf_dist_forward(lo.cuda(), up.cuda(), wd, y, y2, p, p2, G)
    streamed()
    same(y, rl)
    same(y2, ru)
    same(p, rpl)
    same(p2, rpu)
    for K in sorted({2, min(n, 10), min(n, 25)}):
        if K < 2 or K > n:
            continue
        ref = oracle.sort_neuron_forward(x.numpy(), w.numpy(), 0.6, K, groups=G, need_pos=False)
        ext.sort_neuron_forward_nograd(xd, wd, y, G, 0.6, K)
        if B * m * G <= 80 * n:
            streamed()
        np.testing.assert_allclose(y.cpu().numpy(), ref.reshape(B, m * G, 1), rtol=1e-5, atol=1e-6)
        rl, ru = oracle.bound_sort_neuron_forward(lo.numpy(), up.numpy(), w.numpy(), 0.6, K, groups=G)
        ext.bound_sort_neuron_forward(lo.cuda(), up.cuda(), wd, y, y2, G, 0.6, K)
        if B * m * G <= 56 * n:
            streamed()
        np.testing.assert_allclose(y.cpu().numpy(), rl.reshape(B, m * G, 1), rtol=1e-5, atol=1e-6)
        np.testing.assert_allclose(y2.cpu().numpy(), ru.reshape(B, m * G, 1), rtol=1e-5, atol=1e-6)


# batch rows dealt to the workgroups that the device holds at once, one to several rows each, the last one fewer; as many rows as
# workgroups and one more, where two to four rounds of them take over
@pytest.mark.parametrize("B,n,m", [(300, 1024, 70), (33, 700, 1537), (32, 1023, 1536), (255, 5124, 12), (256, 5124, 12), (257, 5121, 12),
                                   (90, 2050, 24), (513, 3100, 10)])
def test_batch_rows_dealt_to_workgroups(oracle, B, n, m):
    from sortnet_amd import _lib, ext
    x, w = _data((B, n, m, 1), "normal")
    xd, wd = x.cuda(), w.cuda()
    y, y2 = (torch.full((B, m, 1), float("nan"), device="cuda") for _ in range(2))
    p = torch.full((B, m, 1), -7, device="cuda", dtype=torch.int32)
    ry, rp = oracle.inf_dist_forward(x.numpy(), w.numpy())
    ext.inf_dist_forward(xd, wd, y, p, 1)
    assert _lib.last_forward_kernel().startswith("row_stream_kernel")
    assert np.array_equal(y.cpu().numpy(), ry) and np.array_equal(p.cpu().numpy(), rp)
    ext.sort_neuron_forward_nograd(xd, wd, y, 1, 0.6, 10)
    assert _lib.last_forward_kernel().startswith("row_stream_kernel")
    ref = oracle.sort_neuron_forward(x.numpy(), w.numpy(), 0.6, 10, need_pos=False)
    np.testing.assert_allclose(y.cpu().numpy(), ref.reshape(B, m, 1), rtol=1e-5, atol=1e-6)   # the same ten products, summed in fp32
    rl, ru = oracle.bound_sort_neuron_forward((x - 0.1).numpy(), (x + 0.1).numpy(), w.numpy(), 0.6, 10)
    ext.bound_sort_neuron_forward((x - 0.1).cuda(), (x + 0.1).cuda(), wd, y, y2, 1, 0.6, 10)
    np.testing.assert_allclose(y.cpu().numpy(), rl.reshape(B, m, 1), rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(y2.cpu().numpy(), ru.reshape(B, m, 1), rtol=1e-5, atol=1e-6)


# one batch row per workgroup: the terms take the weights' registers.  Same products and sums as the kernels with positions, largest
# first: the same bits.  (Few weight rows: several batch rows, each in a workgroup of its own; 16384 and more: more than one round.)
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("B,n,m", [(1, 255, 4), (1, 1023, 9), (1, 1024, 33), (1, 1025, 6), (1, 3071, 5), (1, 3072, 5), (1, 3076, 7), (1, 5119, 6),
                                   (1, 5120, 1030), (1, 5121, 3), (1, 10239, 3), (1, 10240, 5), (9, 4100, 10), (33, 641, 3), (1, 60, 20001),
                                   (1, 64, 33000)])
def test_one_batch_row_has_the_same_bits(B, n, m, kind):
    from sortnet_amd import _lib, ext
    x, w = (t.cuda() for t in _data((B, n, m, 1), kind))
    y, y2 = (torch.full((B, m, 1), float("nan"), device="cuda") for _ in range(2))
    for K in (2, 10, 25):
        pos = torch.empty(K, B, m, 1, device="cuda", dtype=torch.int32)
        ext.sort_neuron_forward_nograd(x, w, y, 1, 0.6, K)
        if m < 20000:
            assert _lib.last_forward_kernel().startswith("row_stream_kernel")
        ext.sort_neuron_forward(x, w, y2, pos, 1, 0.6, K)
        assert np.array_equal(y.cpu().numpy(), y2.cpu().numpy(), equal_nan=True)


@pytest.fixture
def no_sort_tables():
    from sortnet_amd import _lib
    _lib.set_sort_candidate_density(0.0)
    yield
    _lib.set_sort_candidate_density(-1.0)


# layers of more outputs than the limit against tables, where there are none: the kernel that streams still comes before the one
# that forms every term, up to its own limit and not beyond
@pytest.mark.parametrize("B,n,m,streams,bounds", [(100, 639, 630, True, True), (150, 500, 500, True, False), (40, 1657, 1659, True, True),
                                                  (20, 3333, 3334, True, False), (151, 500, 500, False, False)])
def test_layers_without_tables(oracle, no_sort_tables, B, n, m, streams, bounds):
    from sortnet_amd import _lib, ext
    x, w = _data((B, n, m, 1), "ties" if B == 100 else "normal")
    xd, wd = x.cuda(), w.cuda()
    y, y2 = (torch.full((B, m, 1), float("nan"), device="cuda") for _ in range(2))
    ext.sort_neuron_forward_nograd(xd, wd, y, 1, 0.6, 10)
    assert _lib.last_forward_kernel().startswith("row_stream_kernel") == streams
    rows = slice(0, B, 7)   # (an output depends on its own row alone)
    ref = oracle.sort_neuron_forward(x[rows].contiguous().numpy(), w.numpy(), 0.6, 10, need_pos=False)
    np.testing.assert_allclose(y[rows].cpu().numpy(), ref.reshape(-1, m, 1), rtol=1e-5, atol=1e-6)   # ten products, summed in fp32
    ext.bound_sort_neuron_forward((x - 0.1).cuda(), (x + 0.1).cuda(), wd, y, y2, 1, 0.6, 10)
    assert _lib.last_forward_kernel().startswith("row_stream_kernel") == bounds
    rl, ru = oracle.bound_sort_neuron_forward((x[rows] - 0.1).contiguous().numpy(), (x[rows] + 0.1).contiguous().numpy(), w.numpy(), 0.6, 10)
    np.testing.assert_allclose(y[rows].cpu().numpy(), rl.reshape(-1, m, 1), rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(y2[rows].cpu().numpy(), ru.reshape(-1, m, 1), rtol=1e-5, atol=1e-6)
