"""Interval bounds on tiles of 2 x 2 outputs that are held to fewer registers: rows and layers that fill no tile, and spatial positions. Values
are maxima of differences: bits equal to those formed by torch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,M,HW", [(100, 785, 301, 1), (64, 2049, 1000, 1), (1, 33, 31, 1), (33, 31, 33, 1), (8, 75, 100, 49), (5, 27, 33, 36)])
def test_bounds(B, N, M, HW):
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = torch.randn(B, N, HW, generator=g, device="cuda"), torch.randn(M, N, generator=g, device="cuda")
    lo, up = x - 0.1, x + 0.1
    got = F.bound_inf_dist(lo, up, w)
    for b in range(0, B, max(1, B // 7)):
        tl, tu = w[:, :, None] - lo[b], up[b] - w[:, :, None]
        assert torch.equal(got[1][b], torch.maximum(tl, tu).amax(1).clamp(min=1e-10))
        assert torch.equal(got[0][b], (-torch.minimum(tl, tu)).amax(1).clamp(min=1e-10))
