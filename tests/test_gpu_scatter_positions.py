"""Scatter backward of layers with several positions per image, whose rows are taken in runs of neighbouring positions, and of both
gradients in one launch: runs that are not whole, one run per image and many, groups, index lists, rows that LDS holds one run or
one row of, against the oracle.  Sums of fp32 values in any order: relative error 1e-5 of the largest entry."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(got, want):
    np.testing.assert_allclose(got.cpu().numpy(), want, rtol=1e-5, atol=1e-5 * max(np.abs(want).max(), 1e-30))


@pytest.mark.parametrize("B,N,M,G,HW", [(3, 27, 17, 1, 900), (5, 6, 4, 2, 2), (2, 700, 33, 1, 3), (4, 130, 9, 1, 5), (3, 300, 40, 2, 33),
                                        (2, 2700, 20, 1, 4), (2, 6200, 5, 1, 4), (70, 12, 10, 1, 8), (1, 12288, 3, 1, 2), (300, 20, 600, 1, 1)])
def test_runs_of_positions(oracle, B, N, M, G, HW):
    from sortnet_amd import ext
    g = torch.Generator().manual_seed(B + N)
    gy, gu = torch.randn(B, M * G, HW, generator=g), torch.randn(B, M * G, HW, generator=g)
    sign = lambda p: p | (torch.randint(0, 2, p.shape, generator=g) << 31).to(torch.int32)   # noqa: E731
    pos = sign(torch.randint(0, N, (B, M * G, HW), generator=g, dtype=torch.int32))
    pos2 = sign(torch.randint(0, N, (B, M * G, HW), generator=g, dtype=torch.int32))
    xs, ws = (B, N * G, HW), (M * G, N)
    new = lambda s: torch.full(s, 7.0, device="cuda")   # noqa: E731
    rgx, rgw = oracle.inf_dist_backward(gy.numpy(), pos.numpy(), xs, ws, G)
    gx, gw, gi = new(xs), new(ws), new(xs)
    ext.inf_dist_backward_input_weight(gy.cuda(), pos.cuda(), gx, gw, G)
    ext.inf_dist_backward_input(gy.cuda(), pos.cuda(), gi, G)
    _check(gx, rgx)
    _check(gw, rgw)
    _check(gi, rgx)
    pos[0, 0, 0] = -1   # no gradient to the lower bound
    rl, ru, rw = oracle.bound_inf_dist_backward(gy.numpy(), gu.numpy(), pos.numpy(), pos2.numpy(), xs, ws, G)
    gl, gup, gw = new(xs), new(xs), new(ws)
    ext.bound_inf_dist_backward_input_weight(gy.cuda(), gu.cuda(), pos.cuda(), pos2.cuda(), gl, gup, gw, G)
    _check(gl, rl)
    _check(gup, ru)
    _check(gw, rw)
    gl, gup = new(xs), new(xs)
    ext.bound_inf_dist_backward_input(gy.cuda(), gu.cuda(), pos.cuda(), pos2.cuda(), gl, gup, G)
    _check(gl, rl)
    _check(gup, ru)


@pytest.mark.parametrize("B,N,M,kn,km,G,HW", [(70, 96, 64, 29, 21, 1, 1), (40, 64, 48, 12, 8, 2, 7), (33, 40, 24, 27, 9, 1, 40)])
def test_index_lists(oracle, B, N, M, kn, km, G, HW):
    from sortnet_amd import ext
    g = torch.Generator().manual_seed(B)
    keep = lambda c, k: torch.rand(-(-B // 32), G, c, generator=g).argsort(-1)[..., :k].sort(-1)[0].to(torch.int32).contiguous()   # noqa: E731
    ci, co = keep(N, kn), keep(M, km)
    gy = torch.randn(B, km * G, HW, generator=g)
    pos = torch.randint(0, kn, (B, km * G, HW), generator=g, dtype=torch.int32)
    xs, ws = (B, kn * G, HW), (M * G, N)
    rgx, rgw = oracle.inf_dist_backward(gy.numpy(), pos.numpy(), xs, ws, G, True, ci.numpy(), co.numpy())
    gx, gw = torch.full(xs, 7.0, device="cuda"), torch.full(ws, 7.0, device="cuda")
    ext.inf_dist_backward_input_weight(gy.cuda(), pos.cuda(), gx, gw, G, ci.cuda(), co.cuda())
    _check(gx, rgx)
    _check(gw, rgw)
