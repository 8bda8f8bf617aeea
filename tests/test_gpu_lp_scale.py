"""l-p distance at powers above 10 whose scale comes from a part of the inputs (layers of at least 2^29 terms): against 64-bit sums, with
operands whose maximum lies outside that part and so far above it that a sum leaves 32 bits, and with undefined and infinite operands.
Bound: the rounding of a term's exponent (at most 127 in size: 2^-18) and that of the sum (a random walk over N terms) are divided by p in
the root; an ulp each of log2 of the largest difference and of the scale (times ln 2, so 2^-23 of log2, at 1e12 forty times what it is at 2)
is not; the root has 2 ulp of its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _lists(g, subs, channels, kept):
    return torch.rand(subs, 1, channels, generator=g, device="cuda").argsort(-1)[..., :kept].sort(-1)[0].to(torch.int32).contiguous()


# dense on narrow tiles (whole and ragged rows), on wide ones, on exact tiles; index lists; just below the size and just above it
@pytest.mark.parametrize("p", [10.5, 24.0, 31.0])
@pytest.mark.parametrize("B,N,M,lists", [(64, 10240, 1024, False), (250, 3072, 1021, False), (67, 9001, 900, False), (128, 5120, 1600, False),
                                         (64, 3200, 2621, False), (64, 3200, 2622, False), (96, 3000, 2513, True)])
@pytest.mark.parametrize("kind", ["", "far", "undefined"])
def test_scale_from_a_part_of_the_inputs(B, N, M, lists, p, kind):
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = torch.randn(B, N, 1, generator=g, device="cuda") * 0.3, torch.randn(M, N + 500 * lists, generator=g, device="cuda")
    ci = _lists(g, B // 32, N + 500, N) if lists else None
    co = _lists(g, B // 32, M, M - 10) if lists else None
    if kind == "far":       # (whole rows and whole samples, and single ones)
        w[3::7, N - 40] = -1e5
        x[5, N // 2], w[M // 2, 7] = 3e4, 1e12
    if kind == "undefined":
        x[3, N - 1], w[11, 5], w[M - 12, N // 3] = float("nan"), float("inf"), float("nan")
    y = (F.norm_dist_dropout(x, w, ci, co, p) if lists else F.norm_dist(x, w, p))[..., 0]
    rtol = (2 ** -18 + 4 * N ** 0.5 * 2 ** -24) / p + 2 ** -22
    for b in range(0, B, 5) if kind != "undefined" else (0, 3, B - 1):
        rows = w if not lists else w[co[b // 32, 0].long()][:, ci[b // 32, 0].long()]
        d = (x[b, None, :, 0].double() - rows.double()).abs()
        top = d.max(1).values
        ref = (d / top[:, None]).pow(p).sum(1).pow(1 / p) * top
        odd = ~torch.isfinite(ref)
        assert torch.equal(torch.isnan(y[b]), odd) and odd.any() == (kind == "undefined" and (b == 3 or not lists or bool(odd.any())))
        bound = rtol + 2 * 2 ** -23 * top.log2().abs().clamp(min=2)
        assert ((y[b].double() - ref).abs() <= bound * ref)[~odd].all()
