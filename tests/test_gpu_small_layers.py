"""Layers that leave most of the device idle: tiles of 32 x 32 outputs, slices of one chunk, few outputs per wavefront in
the position pass, sliced backward, batches that are no multiple of the backward's 32 rows.  l-inf and interval layers
against the oracle bit for bit; l-p against float64 within the rounding of fp32 sums, a ratio's rounding to the power p - 1."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# batch, inputs, outputs, groups, positions: one row over and under a tile, a chunk and a slice of channels
SHAPES = [(33, 1025, 257, 1, 1), (31, 2048, 129, 1, 1), (65, 1000, 1000, 1, 1), (250, 1024, 1021, 1, 1), (40, 4100, 516, 2, 1),
          (9, 300, 310, 1, 4), (26, 5120, 200, 1, 1)]
# the kernel that serves the maxima, the maxima with positions, the bounds and the bounds with positions: layers this small
# are streamed where they are dense, the rest are past the streaming limits on purpose
STREAM, VECTOR, GATHER, GENERAL = "row_stream_kernel", "fwd_kernel_pipe<2,2>", "fwd_kernel_lists<2,2>", "fwd_kernel<2,2>"
KERNELS = {(65, 1000, 1000, 1, 1): (STREAM, STREAM, STREAM, VECTOR), (250, 1024, 1021, 1, 1): (VECTOR,) * 4,
           (9, 300, 310, 1, 4): (GATHER, GATHER, GENERAL, GENERAL),
           (130, 2048, 513, 1, 1): (VECTOR,) * 4, (300, 3072, 129, 1, 1): (VECTOR,) * 4,
           (161, 1025, 700, 1, 1): (GATHER, GATHER, GENERAL, GENERAL), (97, 4100, 516, 2, 1): (GATHER, GATHER, GENERAL, GENERAL),
           (32, 33, 129, 1, 4097): ("fwd_kernel<4,8>", "fwd_kernel_lists<2,8>", "fwd_kernel<4,8>", "fwd_kernel<4,4>")}


def _data(shape):
    B, n, m, G, hw = shape
    g = torch.Generator().manual_seed(B + n + m)
    return torch.randn(B, n, hw, generator=g), torch.randn(m, n // G, generator=g), torch.randn(B, m, hw, generator=g)


def _served_by(name):
    from sortnet_amd import _lib
    assert _lib.last_forward_kernel().startswith(name), _lib.last_forward_kernel()


@pytest.mark.parametrize("shape", SHAPES + [s for s in KERNELS if s not in SHAPES], ids=lambda s: "x".join(map(str, s)))
def test_maxima_positions_and_bounds(oracle, shape):
    from sortnet_amd import ext
    kernels = KERNELS.get(shape, (STREAM,) * 4)
    B, n, m, G, hw = shape
    n, m = n // G * G, m // G * G
    x, w, _ = _data((B, n, m, G, hw))
    x[0, 3], w[1, 2] = float("nan"), float("inf")     # undefined terms never win, infinite ones do
    xd, wd = x.cuda(), w.cuda()
    y, y2, p, p2 = (torch.empty(B, m, hw, device="cuda", dtype=t) for t in (torch.float32,) * 2 + (torch.int32,) * 2)

    def same(got, ref):
        assert np.array_equal(got.cpu().numpy(), np.asarray(ref).reshape(tuple(got.shape)), equal_nan=True)

    ry, rp = oracle.inf_dist_forward(x.numpy(), w.numpy(), G)
    ext.inf_dist_forward_nograd(xd, wd, y, G)
    _served_by(kernels[0])
    same(y, ry)
    ext.inf_dist_forward(xd, wd, y.zero_(), p, G)
    _served_by(kernels[1])
    same(y, ry)
    same(p, rp)
    vector = "fwd_kernel_pipe<" if n // G % 4 == 0 and hw == 1 else "fwd_kernel<"
    for mode in (oracle.MASK_FACTORED, oracle.MASK_TERM):
        ry, rp = oracle.masked_inf_dist_forward(x.numpy(), w.numpy(), 0.4, 11, mode, groups=G)
        for pos in (None, p):
            ext.masked_inf_dist_forward(xd, wd, y.zero_(), pos, G, 0.4, 11, mode)
            streamed = mode == oracle.MASK_FACTORED and hw == 1 and B * m * n // G <= 3 << 24
            _served_by(STREAM if streamed else vector)
            same(y, ry)
        same(p, rp)
    x[0, 3], w[1, 2] = 0.25, 0.5
    lo, up = x - 0.1, x + 0.1
    rl, ru, rpl, rpu = oracle.bound_inf_dist_forward(lo.numpy(), up.numpy(), w.numpy(), G)
    ext.bound_inf_dist_forward_nograd(lo.cuda(), up.cuda(), w.cuda(), y, y2, G)
    _served_by(kernels[2])
    same(y, rl)
    same(y2, ru)
    ext.bound_inf_dist_forward(lo.cuda(), up.cuda(), w.cuda(), y, y2, p, p2, G)
    _served_by(kernels[3])
    same(y, rl)
    same(y2, ru)
    same(p, rpl)
    same(p2, rpu)


@pytest.mark.parametrize("p", [8.0, 9.5, 24.0, 100.0])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s[3] == 1], ids=lambda s: "x".join(map(str, s)))
def test_lp_values_and_gradients(shape, p):
    from sortnet_amd import functional as F
    B, n, m, _, hw = shape
    x, w, gy = _data(shape)
    xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
    y = F.norm_dist(xd, wd, p)
    # rows that are not loaded by 16 bytes go online at large p, on tiles that are not narrowed
    _served_by(VECTOR if n % 4 == 0 and hw == 1 else GATHER if p <= 10 else "fwd_kernel_lists<2,8>")
    gx, gw = torch.autograd.grad(y, [xd, wd], gy.cuda())
    ry, rx, rw = torch.empty(B, m, hw).double(), torch.zeros(B, n, hw).double(), torch.zeros(m, n).double()
    wd64 = w.cuda().double()
    for b in range(B):
        for k in range(hw):
            d = x[b, :, k].cuda().double() - wd64
            top = d.abs().amax(1, keepdim=True)
            v = top[:, 0] * ((d.abs() / top) ** p).sum(1) ** (1 / p)
            u = gy[b, :, k].cuda().double()[:, None] * d.sign() * (d.abs() / v[:, None]) ** (p - 1)
            ry[b, :, k], rx[b, :, k] = v.cpu(), u.sum(0).cpu()
            rw -= u.cpu()
    for got, ref in ((y.detach(), ry), (gx, rx), (gw, rw)):
        # p roundings of a ratio (6e-8 each, its error taken to the power p - 1) and the fp32 sums
        assert (got.cpu().double() - ref).norm() <= max(1e-5, 1e-6 * p) * ref.norm()


@pytest.mark.parametrize("B,n,m", [(33, 200, 90), (250, 1025, 515), (26, 3000, 40)])
def test_index_lists_match_the_dense_layer(B, n, m):
    """Lists that keep everything, and the same layer without lists: same values, positions and gradients up to the order of
    the sums."""
    from sortnet_amd import functional as F
    x, w, gy = (t.cuda() for t in _data((B, n, m, 1, 1)))
    subs = -(-B // 32)
    ci, co = (torch.arange(c, device="cuda", dtype=torch.int32).expand(subs, 1, c).contiguous() for c in (n, m))
    for p in (8.0, 24.0, float("inf")):
        a = [x.clone().requires_grad_(), w.clone().requires_grad_()]
        y = F.norm_dist(*a, p)
        b = [x.clone().requires_grad_(), w.clone().requires_grad_()]
        z = F.norm_dist_dropout(*b, ci, co, p)
        _served_by(GATHER)
        for u, v in zip([y, *torch.autograd.grad(y, a, gy)], [z, *torch.autograd.grad(z, b, gy)]):
            assert (u - v).norm() <= 3e-5 * v.norm()
