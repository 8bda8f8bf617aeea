"""Gradients of the l-p distance (sd_norm_dist_backward_input[_weight]) where the kernel from scalar registers can go wrong:
tiles of 32 rows and 64 inputs and chunks of 4 channels that are not whole, positions side by side in runs of every length,
slices merged from planes, batches of several workgroups' tiles, and outputs too small or too large to be raised to the power
p - 1 by themselves, next to ordinary ones.  Sums of fp32 products in any order: relative error 1e-5 of the largest entry."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(got, want):
    np.testing.assert_allclose(got.cpu().numpy(), want, rtol=1e-5, atol=1e-5 * np.abs(want).max())


def _both(oracle, x, w, gy, p, G=1, ci=None, co=None):
    from sortnet_amd import ext
    lists = ci is not None
    n = lambda t: None if t is None else t.numpy()   # noqa: E731
    ry = oracle.norm_dist_forward(x.numpy(), w.numpy(), p, G, n(ci), n(co))
    rgx, rgw = oracle.norm_dist_backward(gy.numpy(), x.numpy(), w.numpy(), ry, p, G, True, n(ci), n(co))
    dev = torch.device("cuda:0")
    xd, wd, gd, yd = x.to(dev), w.to(dev), gy.to(dev), torch.from_numpy(ry).to(dev)
    lists = (ci.to(dev), co.to(dev)) if lists else (None, None)
    gx, gw, gi = torch.full_like(xd, 7), torch.full_like(wd, 7), torch.full_like(xd, 7)
    ext.norm_dist_backward_input_weight(gd, xd, wd, yd, gx, gw, G, p, *lists)
    ext.norm_dist_backward_input(gd, xd, wd, yd, gi, G, p, *lists)
    _check(gx, rgx)
    _check(gw, rgw)
    _check(gi, rgx)


@pytest.mark.parametrize("p", [2.0, 7.0, 8.0, 9.0, 12.7])
@pytest.mark.parametrize("B,N,M,G,HW", [
    (1, 1, 1, 1, 1), (33, 65, 5, 1, 1), (130, 700, 67, 1, 1), (31, 64, 1021, 1, 1), (160, 512, 130, 2, 1), (3, 27, 17, 1, 49),
    (20, 75, 33, 1, 3), (9, 144, 20, 1, 40), (40, 130, 12, 2, 2), (2, 27, 48, 1, 1024), (129, 2048, 260, 1, 1)])
def test_edges_of_tiles(oracle, p, B, N, M, G, HW):
    g = torch.Generator().manual_seed(B * 7 + N)
    x, gy = torch.randn(B, N * G, HW, generator=g), torch.randn(B, M * G, HW, generator=g)
    _both(oracle, x, torch.randn(M * G, N, generator=g) * 0.4, gy, p, G)


@pytest.mark.parametrize("p", [2.0, 8.0, 9.0])
@pytest.mark.parametrize("HW", [1, 5])
def test_outputs_of_any_scale(oracle, p, HW):
    """Rows and channels from 1e-4 to 1e4 times the ordinary scale: chunks that form ratios beside chunks that form products."""
    g = torch.Generator().manual_seed(3)
    B, N, M = 70, 130, 44
    scale = torch.ones(B, 1, 1)
    scale[5], scale[40:43], scale[69] = 1e-4, 1e4, 1e-3
    x, gy = torch.randn(B, N, HW, generator=g) * scale, torch.randn(B, M, HW, generator=g)
    w = torch.randn(M, N, generator=g) * 1e-5
    w[9], w[20:22] = 1e4, 300.0
    gy[:, 13] = 0
    _both(oracle, x, w, gy, p)
    gy[:, 30] *= 1e-30
    _both(oracle, x[:33].contiguous(), w, gy[:33].contiguous(), p)


@pytest.mark.parametrize("B,N,M,kn,km,G,HW", [(70, 96, 64, 67, 21, 1, 1), (33, 130, 44, 100, 33, 2, 1), (64, 40, 24, 27, 9, 1, 3)])
def test_index_lists(oracle, B, N, M, kn, km, G, HW):
    g = torch.Generator().manual_seed(B)
    keep = lambda c, k: torch.rand(-(-B // 32), G, c, generator=g).argsort(-1)[..., :k].sort(-1)[0].to(torch.int32).contiguous()   # noqa: E731
    ci, co = keep(N, kn), keep(M, km)
    x, gy = torch.randn(B, kn * G, HW, generator=g), torch.randn(B, km * G, HW, generator=g)
    for p in (3.0, 8.0, 10.5):
        _both(oracle, x, torch.randn(M * G, N, generator=g), gy, p, G, ci, co)


# Workgroups of four batch tiles from 1024 (tile, 64 inputs, group) triples on.  A tile behind the batch has inputs of no row: here row 0 is so
# far from the weights that the products of a factor 0 with powers of its distances would be undefined.
@pytest.mark.parametrize("p,far", [(2.0, 1e30), (6.0, 1e16), (8.0, 1e10), (9.0, 1e8), (17.3, 1e8)])
def test_tiles_behind_the_batch(oracle, p, far):
    g = torch.Generator().manual_seed(6)
    B, N, M = 336, 6001, 6
    x, gy = torch.randn(B, N, 1, generator=g), torch.randn(B, M, 1, generator=g)
    x[0, 7], x[0, 5990] = far, -far
    _both(oracle, x, torch.randn(M, N, generator=g) * 0.4, gy, p)


@pytest.mark.parametrize("p", [2.0, 3.0])
def test_input_gradients_of_large_batches(p):
    """Sums over the output channels are cut into as many slices as by the general kernel (three here): the error of grad_input is not above
    (by more than its sampling, a tenth) that of 32-bit sums over slices of 344 channels."""
    from sortnet_amd import ext
    g = torch.Generator(device="cuda").manual_seed(8)
    B, N, M = 8192, 2048, 1024
    x, w, gy = (torch.randn(*s, generator=g, device="cuda") for s in ((B, N, 1), (M, N), (B, M, 1)))
    y, gx, gw = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(w)
    ext.norm_dist_forward(x, w, y, 1, p)
    ext.norm_dist_backward_input_weight(gy, x, w, y, gx, gw, 1, p)
    rows = slice(None, None, 512)
    xs, gs, ys = x[rows, :, 0], gy[rows, :, 0], y[rows, :, 0].double()
    exact, parts = torch.zeros_like(xs, dtype=torch.float64), []
    for m in range(M):
        if m % 344 == 0:
            parts.append(torch.zeros_like(xs))
        d = xs - w[m]
        k = gs[:, m, None].double() * ys[:, m, None] ** (1 - p)
        e = xs.double() - w[m].double()
        exact += k * e * e.abs() ** (p - 2)
        t = d.abs() * k.float() if p == 3.0 else k.float()
        parts[-1] = (parts[-1].double() + t.double() * d.double()).float()   # one fused multiply-add
    error = lambda got: float((got.double() - exact).norm() / exact.norm())   # noqa: E731
    assert error(gx[rows, :, 0]) <= 1.1 * error(sum(parts))


@pytest.mark.parametrize("p,B,N,M,channels", [(2.0, 167, 62, 883, 16), (1.0, 16, 164, 1417, 8)])
def test_input_gradients_of_fine_slices(p, B, N, M, channels):
    """Small layers, cut into slices of four output channels: the error of grad_input is not above (by more than its sampling, a tenth) that of
    32-bit sums over slices of `channels`, as the general kernel cuts them, merged a quarter of the slices at a time."""
    from sortnet_amd import ext
    g = torch.Generator(device="cuda").manual_seed(8)
    x, w, gy = (torch.randn(*s, generator=g, device="cuda") for s in ((B, N, 1), (M, N), (B, M, 1)))
    y, gx, gw = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(w)
    ext.norm_dist_forward(x, w, y, 1, p)
    ext.norm_dist_backward_input_weight(gy, x, w, y, gx, gw, 1, p)
    exact, parts = torch.zeros(B, N, device="cuda", dtype=torch.float64), []
    for m in range(M):
        if m % channels == 0:
            parts.append(torch.zeros(B, N, device="cuda"))
        d = x[:, :, 0] - w[m]
        e = x[:, :, 0].double() - w[m].double()
        u = gy[:, m].double() * (e / y[:, m].double() if p == 2.0 else e.sign())
        exact += u
        t = gy[:, m] / y[:, m] if p == 2.0 else gy[:, m]
        parts[-1] = (parts[-1].double() + t.double() * (d if p == 2.0 else d.sign()).double()).float()   # one fused multiply-add
    per = -(-len(parts) // 4)
    quarters = [sum(parts[q * per:(q + 1) * per]) for q in range(4)]
    error = lambda got: float((got.double() - exact).norm() / exact.norm())   # noqa: E731
    assert error(gx[:, :, 0]) <= 1.1 * error(quarters[0] + quarters[1] + quarters[2] + quarters[3])


@pytest.mark.parametrize("p", [2.0, 3.0, 4.0, 5.0, 6.0, 7.0, 8.0, 9.0])
@pytest.mark.parametrize("gscale", [1e-30, 1.0, 1e30])
def test_edges_of_the_ranges(oracle, p, gscale):
    """Every row at a scale of its own, from far below to far above the limits of the product form (2^(-70 / (p-1)) to 2^(120 / (p-1)) for an
    output); gradients are so of ratios, whatever the scale."""
    g = torch.Generator().manual_seed(int(p))
    B, N, M = 64, 70, 40
    reach = 124 / (p - 1)
    scale = 2.0 ** torch.linspace(-max(80 / (p - 1), 8), min(reach, 110), 32).repeat_interleave(2).view(B, 1, 1)
    x, gy = torch.randn(B, N, 1, generator=g) * scale, torch.randn(B, M, 1, generator=g) * gscale
    _both(oracle, x, torch.randn(M, N, generator=g) * 1e-4, gy, p)
    tile = x[30:31] * torch.randn(33, N, 1, generator=g)   # a whole tile and a row at one scale, and with zeros among the gradients
    gy[:33, ::3] = 0
    _both(oracle, tile.contiguous(), torch.randn(M, N, generator=g) * 1e-4, gy[:33].contiguous(), p)


@pytest.mark.parametrize("p,xscale,gscale", [(2.0, 1000.0, 1.0), (8.0, 1000.0, 1.0), (8.0, 1.0, 1e-30)])
def test_time_follows_the_sizes(p, xscale, gscale):
    """Large outputs, and gradients that are almost nothing in one channel of four, take at most 1.6 times as long as ordinary ones (the
    loop that forms ratios: 1.25; row by row it took 2.7)."""
    from sortnet_amd import ext
    g = torch.Generator(device="cuda").manual_seed(9)
    x, w, gy = (torch.randn(*s, generator=g, device="cuda") for s in ((512, 5120, 1), (512, 5120), (512, 512, 1)))
    y, gx, gw = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(w)

    def least(x, w, gy):
        ext.norm_dist_forward(x, w, y, 1, p)
        times = []
        for _ in range(12):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            ext.norm_dist_backward_input_weight(gy, x, w, y, gx, gw, 1, p)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    ordinary = least(x, w, gy)
    gy[:, ::4] *= gscale
    assert least(x * xscale, w * xscale, gy) <= 1.6 * ordinary


@pytest.mark.parametrize("p,B,N,M,HW,both,scalars", [
    (8.0, 8, 1024, 1024, 1, True, False), (8.0, 9, 1024, 1024, 1, True, True), (8.0, 3, 3072, 2800, 1, True, True), (8.0, 8, 5120, 5120, 1, False, False),
    (8.0, 17, 640, 640, 1, False, False), (8.0, 33, 1024, 1024, 1, False, True), (2.0, 8, 27, 64, 2, True, False), (8.0, 9, 27, 64, 2, True, True),
    (8.0, 64, 288, 256, 4, False, False), (8.0, 32, 288, 128, 16, False, True), (17.3, 4, 1024, 1024, 1, True, False), (17.3, 33, 2001, 2000, 1, True, False),
    (17.3, 33, 800, 800, 1, True, True), (17.3, 250, 1024, 1024, 1, True, True), (17.3, 64, 800, 800, 1, True, False), (17.3, 128, 800, 256, 4, True, False)])
def test_which_kernel(oracle, p, B, N, M, HW, both, scalars):
    """Few rows, and small layers where only the gradient of the inputs is asked for, go through the general kernel."""
    from torch.profiler import ProfilerActivity, profile
    from sortnet_amd import ext
    g = torch.Generator().manual_seed(B)
    x, w, gy = (torch.randn(*s, generator=g) for s in ((B, N, HW), (M, N), (B, M, HW)))
    y = torch.empty(B, M, HW, device="cuda")
    xd, wd, gd = x.cuda(), w.cuda(), gy.cuda()
    ext.norm_dist_forward(xd, wd, y, 1, p)
    gx, gw = torch.empty_like(xd), torch.empty_like(wd)
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        if both:
            ext.norm_dist_backward_input_weight(gd, xd, wd, y, gx, gw, 1, p)
        else:
            ext.norm_dist_backward_input(gd, xd, wd, y, gx, 1, p)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events()]
    assert any("lp_grad_kernel" in n for n in names) == scalars and any("lp_bwd_kernel" in n for n in names) != scalars, names
    if B * N * M * HW < 1 << 25:
        rgx, rgw = oracle.norm_dist_backward(gy.numpy(), x.numpy(), w.numpy(), y.cpu().numpy(), p)
        _check(gx, rgx)
        if both:
            _check(gw, rgw)


def _against_64(x, w, gy, p):
    """Both gradients on the GPU against 64-bit sums there, channel by channel; y as a forward in 64 bits gives it."""
    from sortnet_amd import ext
    x, w, gy = x.cuda(), w.cuda(), gy.cuda()
    y = torch.empty_like(gy)
    gx, gw = torch.full_like(x, 7), torch.full_like(w, 7)
    rx, rw = torch.zeros_like(x, dtype=torch.float64), torch.zeros_like(w, dtype=torch.float64)
    for m in range(w.shape[0]):
        d = x.double() - w[m, None, :, None].double()
        y[:, m] = (d.abs() ** p).sum(1) ** (1 / p)
        u = gy[:, m, None].double() * d.sign() * (d.abs() / y[:, m, None].double()) ** (p - 1)
        rx += u
        rw[m] = -u.sum((0, 2))
    ext.norm_dist_backward_input_weight(gy, x, w, y, gx, gw, 1, p)
    _check(gx, rx.cpu().numpy())
    _check(gw, rw.cpu().numpy())


@pytest.mark.parametrize("p", [2.0, 8.0, 9.0])
@pytest.mark.parametrize("B,N,M,HW,odd", [
    (337, 6016, 10, 1, False), (337, 6016, 10, 1, True),      # 11 tiles of three workgroups, the last one's with one row; chunks that form ratios in it
    (43, 27, 17, 784, False), (43, 27, 17, 784, True),        # positions, 1054 tiles
    (128, 16500, 9, 1, True), (101, 16500, 9, 1, False),      # the whole batch in a workgroup
    (79, 3, 577, 1009, True)])                                # more tiles than the tables of one launch hold
def test_workgroups_of_four_tiles(p, B, N, M, HW, odd):
    assert -(-N // 64) * -(-B * HW // 32) >= 1024   # (batch tile, 64 inputs) pairs from which on four tiles make a workgroup
    g = torch.Generator().manual_seed(B + N)
    x, w, gy = torch.randn(B, N, HW, generator=g), torch.randn(M, N, generator=g), torch.randn(B, M, HW, generator=g)
    if odd:   # outputs outside the product form's range in one tile of a workgroup, and in the chunks of one channel
        x[B // 2] *= 1e9 if p > 2 else 1e36
        w[M // 2] *= 1e-9
        x[B // 3] *= 1e-9
    _against_64(x, w, gy, p)


@pytest.mark.parametrize("p", [3.0, 17.3])
def test_other_shapes_with_many_tiles(oracle, p):
    """Groups and four tiles to a workgroup at other powers; index lists over more than one round of wavefronts."""
    g = torch.Generator().manual_seed(2)
    _both(oracle, torch.randn(333, 2 * 3010, 1, generator=g), torch.randn(10, 3010, generator=g), torch.randn(333, 10, 1, generator=g), p, 2)
    keep = lambda c, k: torch.rand(18, 1, c, generator=g).argsort(-1)[..., :k].sort(-1)[0].to(torch.int32).contiguous()   # noqa: E731
    x, gy = torch.randn(570, 3900, 1, generator=g), torch.randn(570, 9, 1, generator=g)
    _both(oracle, x, torch.randn(14, 5000, generator=g), gy, p, 1, keep(5000, 3900), keep(14, 9))
