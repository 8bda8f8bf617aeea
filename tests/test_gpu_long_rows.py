"""Tile kernels at the edges of their staging: chunks that end behind the row (with and without slices), rows and channels that do not fill a
tile, and rows so long that a tile's byte offsets leave 32 bits, which the general kernel takes.  Maxima and positions are exact.  Sums are those of terms that are 0 or 1, exact in 32 bits inside a slice (at most 2^24 terms); up
to 64 slices are added, half an ulp each, which the root halves, and the root itself has 2 ulp: 2^-19 at most.  (Random terms would not do:
a sum of 5e5 of them is 1.9e-4 off in 32 bits, by the order of the additions alone.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,M,HW,kernel", [
    (33, 4, 35, 1, None), (34, 36, 33, 1, None), (130, 1004, 701, 1, "fwd_kernel_pipe"), (257, 2076, 170, 1, "fwd_kernel_pipe"), (131, 1003, 700, 1, "fwd_kernel_lists"),
    (9, 2701, 65, 4, "fwd_kernel_lists"), (65, 29, 31, 3, "fwd_kernel_lists"), (2, 3000004, 3, 1, "fwd_kernel_pipe"),
    (2, 32000004, 3, 1, "fwd_kernel<"), (2, 8000003, 3, 4, "fwd_kernel_lists"), (2, 80000000, 2, 2, "fwd_kernel<")])
def test_ends_of_rows(B, N, M, HW, kernel):
    from sortnet_amd import _lib, ext
    g = torch.Generator(device="cuda").manual_seed(B + N)
    x, w = torch.rand(B, N, HW, device="cuda", generator=g), torch.randn(M, N, device="cuda", generator=g)
    y, pos = torch.empty(B, M, HW, device="cuda"), torch.empty(B, M, HW, device="cuda", dtype=torch.int32)
    ext.inf_dist_forward(x, w, y, pos, 1)
    if kernel:
        assert _lib.last_forward_kernel().startswith(kernel), _lib.last_forward_kernel()
    y2, y3 = torch.empty_like(y), torch.empty_like(y)
    ext.inf_dist_forward_nograd(x, w, y2, 1)
    x01, w01 = (x < 0.5).float(), (w < 0.0).float()
    ext.norm_dist_forward(x01, w01, y3, 1, 2.0)
    for m in range(0, M, 1 + M // 8):
        d = x - w[m].view(1, N, 1)
        big, at = d.abs().max(1)
        assert torch.equal(y[:, m], big) and torch.equal(y2[:, m], big)
        assert torch.equal(pos[:, m] & 0x7fffffff, at.int())
        assert torch.equal(pos[:, m] < 0, d.gather(1, at.unsqueeze(1)).squeeze(1) < 0)
        ref = (x01 != w01[m].view(1, N, 1)).sum(1).double().sqrt()
        torch.testing.assert_close(y3[:, m].double(), ref, rtol=2 ** -19, atol=2e-10)   # (no term: the 1e-10 that a distance is at least)
