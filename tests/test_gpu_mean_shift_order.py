"""Mean shift: the order in which a channel's values are added, the same in one launch and in two. Without positions every 16th sample, then
the 16 sums; with positions every 1024th value, then the 1024 sums. Formed in 32 bits on the CPU; equal bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C,HW", [(1, 3, 1), (15, 63, 1), (128, 70, 1), (129, 65, 1), (512, 77, 1), (513, 77, 1), (1, 5, 4), (129, 2100, 4), (512, 515, 4),
                                    (8, 9, 64), (300, 60, 64), (33, 9, 8), (40, 40, 3), (600, 20, 4), (256, 512, 4)])
def test_sums_in_a_stated_order(B, C, HW):
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(B + C)
    x = torch.randn(B, C, HW, device="cuda", generator=g) + 3
    running = torch.randn(C, device="cuda", generator=g)
    before = running.cpu()
    y, mean = F.mean_shift(x, running, 0.1)
    slots, n = 16 if HW == 1 else 1024, B * HW
    values = torch.zeros((n + slots - 1) // slots * slots, C)
    values[:n] = x.cpu().permute(0, 2, 1).reshape(n, C)
    sums = torch.zeros(slots, C)
    for part in values.view(-1, slots, C):
        sums = sums + part
    total = torch.zeros(C)
    for part in sums:
        total = total + part
    want = total / n
    assert torch.equal(mean.cpu(), want)
    assert torch.equal(y.cpu(), x.cpu() - want.view(1, -1, 1))
    tenth = torch.tensor(0.1)
    assert torch.equal(running.cpu(), (1 - tenth) * before + tenth * want)
