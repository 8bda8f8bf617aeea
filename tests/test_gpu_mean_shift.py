"""Mean shift in one launch (up to 512 samples, 1 or 4, 8 .. 64 positions) and in two: rows that fill no wavefront, columns that fill no workgroup,
channels of fewer and of more than 1024 values.  Against 64-bit means: n additions of values of size a, half an ulp of their sum each."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C,HW", [(1, 1, 1), (15, 63, 1), (17, 65, 1), (128, 1000, 1), (129, 130, 1), (512, 77, 1), (513, 77, 1), (1, 5, 4), (16, 17, 4),
                                    (128, 33, 4), (129, 2100, 4), (512, 515, 4), (7, 3, 64), (8, 9, 64), (300, 60, 64), (33, 9, 8), (40, 40, 3), (5, 70, 2),
                                    (31, 1100, 32), (500, 131, 16)])
def test_mean_shift(B, C, HW):
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(B + C)
    x = torch.randn(B, C, HW, device="cuda", generator=g) + 3
    x.requires_grad_()
    running = torch.randn(C, device="cuda", generator=g)
    before, gy = running.double(), torch.randn(B, C, HW, device="cuda", generator=g)
    y, mean = F.mean_shift(x, running, 0.1)
    y.backward(gy)
    bound = (B * HW + 4) * 2 ** -24
    for got, at, values in ((y, mean, x.detach()), (x.grad, None, gy)):
        size = values.double().abs().mean((0, 2), keepdim=True)
        ref = values.double().mean((0, 2), keepdim=True)
        assert ((got.double() - (values.double() - ref)).abs() <= bound * size + 2 ** -23 * (values.double().abs() + size)).all()
        if at is not None:
            assert ((at.double() - ref[0, :, 0]).abs() <= bound * size[0, :, 0]).all()
            assert ((running.double() - (0.9 * before + 0.1 * ref[0, :, 0])).abs() <= (bound + 2 ** -21) * (size[0, :, 0] + before.abs())).all()
