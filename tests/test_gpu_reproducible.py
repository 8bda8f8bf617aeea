"""l-p gradients that are the same bits in every call: sums of at most two addends per element, or merged in a fixed order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(B, n, m, G, hw, alike=False):
    g = torch.Generator().manual_seed(B + n + m)
    x = torch.rand(B, n, hw, generator=g)
    if alike:
        x = x[:1] + 0.01 * x
    return x.cuda(), torch.randn(m, n // G, generator=g).cuda(), torch.randn(B, m, hw, generator=g).cuda()


def _differing(x, w, gy, p, G, both):
    """How many elements of the gradients came out as other bits in any of six more calls."""
    from sortnet_amd import ext
    y, gx, gw = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(w)
    ext.norm_dist_forward(x, w, y, G, p)

    def run():
        if both:
            ext.norm_dist_backward_input_weight(gy, x, w, y, gx.fill_(7), gw.fill_(7), G, p)
        else:
            ext.norm_dist_backward_input(gy, x, w, y, gx.fill_(7), G, p)

    run()
    rx, rw, dx, dw = gx.clone(), gw.clone(), 0, 0
    for _ in range(6):
        run()
        dx += int((gx != rx).sum())
        dw += int((gw != rw).sum()) if both else 0
    return dx, dw, rx, rw


# outputs per group below 192; one and two channels past a chunk, one row past a tile, groups, positions, odd planes
@pytest.mark.parametrize("B,n,m,G,hw,p", [(33, 785, 100, 1, 1, 8.0), (64, 1024, 150, 1, 1, 8.0), (16, 64, 9, 1, 1, 3.0), (1, 30, 10, 1, 1, 5.5),
                                          (64, 600, 380, 2, 1, 5.5), (32, 301, 150, 1, 4, 8.0), (250, 3072, 191, 1, 1, 9.0)])
def test_grad_input_of_few_outputs(B, n, m, G, hw, p):
    x, w, gy = _layer(B, n, m, G, hw)
    for both in (True, False):
        assert _differing(x, w, gy, p, G, both)[0] == 0


def test_grad_input_of_index_lists():
    from sortnet_amd import ext
    g = torch.Generator().manual_seed(3)
    x, w, gy = torch.rand(70, 96, 1, generator=g).cuda(), torch.randn(200, 130, generator=g).cuda(), torch.randn(70, 150, 1, generator=g).cuda()
    ci, co = (torch.rand(3, 1, c, generator=g).argsort(-1)[..., :k].sort(-1)[0].to(torch.int32).cuda() for c, k in ((130, 96), (200, 150)))
    y, gx, gw = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(w)
    ext.norm_dist_forward(x, w, y, 1, 8.0, ci, co)
    seen = []
    for _ in range(6):
        ext.norm_dist_backward_input_weight(gy, x, w, y, gx, gw, 1, 8.0, ci, co)
        seen.append(gx.clone())
    assert all(torch.equal(s, seen[0]) for s in seen)


@pytest.mark.parametrize("alike", [True, False])
@pytest.mark.parametrize("B,n,m,p", [(97, 1024, 515, 24.0), (250, 3072, 500, 24.0), (250, 3072, 1021, 100.0), (512, 600, 600, 100.0),
                                     (1025, 1024, 1024, 120.0), (70, 64, 3, 200.0)])
def test_both_gradients_at_large_p(B, n, m, p, alike):
    """Where tables or the fused kernel would serve a larger layer; the batch of 1025 is taken in several launches."""
    from sortnet_amd import _lib
    x, w, gy = _layer(B, n, m, 1, 1, alike)
    large = B * n * m >= 1 << 30
    try:
        if large:      # without tables, which add to grad_input in any order from three tiles of weight rows on
            _lib.set_lp_candidate_density(0)
        dx, dw, gx, gw = _differing(x, w, gy, p, 1, True)
    finally:
        _lib.set_lp_candidate_density(-1)
    assert (dx, dw) == (0, 0)
    assert large or _differing(x, w, gy, p, 1, False)[0] == 0
    # against float64: a ratio's rounding (6e-8) to the power p - 1, and sums in fp32
    rx, rw = torch.zeros(B, n, dtype=torch.float64), torch.zeros(m, n, dtype=torch.float64)
    rx, rw, w64 = rx.cuda(), rw.cuda(), w.double()
    for b in range(B):
        d = x[b, :, 0].double() - w64
        top = d.abs().amax(1, keepdim=True)
        v = top * ((d.abs() / top) ** p).sum(1, keepdim=True) ** (1 / p)
        u = gy[b, :, 0].double()[:, None] * d.sign() * (d.abs() / v) ** (p - 1)
        rx[b] = u.sum(0)
        rw -= u
    for got, ref in ((gx[..., 0], rx), (gw, rw)):
        assert (got.double() - ref).norm() <= 1e-6 * p * ref.norm()
