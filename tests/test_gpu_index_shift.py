"""Mean shift of compacted layers in one launch: sub-batches one over and under the wavefronts of a workgroup, channels over
and under its 64, lists in any order, channels that no sub-batch kept."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,G,cnt,Cg,HW", [(1, 1, 1, 1, 1), (33, 2, 5, 7, 1), (32, 1, 64, 65, 1), (512, 1, 100, 130, 1), (545, 3, 40, 64, 1),
                                           (4096, 1, 9, 12, 1), (4097, 1, 9, 12, 1), (70, 2, 6, 9, 3)])
def test_mean_shift_of_compacted_layers(B, G, cnt, Cg, HW):
    from sortnet_amd import functional as F
    g = torch.Generator().manual_seed(B + cnt)
    S = -(-B // 32)
    index = torch.rand(S, G, Cg, generator=g).argsort(-1)[..., :cnt].to(torch.int32)     # in no order
    x = torch.randn(B, G * cnt, HW, generator=g)
    running = torch.randn(G * Cg, generator=g)
    chan = (index.long() + torch.arange(G)[None, :, None] * Cg).reshape(S, G * cnt).repeat_interleave(32, 0)[:B]
    total = torch.zeros(G * Cg).double().index_add_(0, chan.flatten(), x.double().sum(2).flatten())
    seen = torch.zeros(G * Cg).double().index_add_(0, chan.flatten(), torch.ones(B * G * cnt).double())
    mean = total / (seen * HW).clamp_(min=1e-10)
    rd = running.cuda()
    y, m = F.mean_shift_index(x.cuda(), index.cuda(), G * Cg, rd, 0.1)
    # sums of up to B * HW values of size 1 in fp32
    bar = 1e-6 * (B * HW) ** 0.5 / max(1, int(seen[seen > 0].min()) ** 0.5) + 1e-6
    assert (m.cpu().double() - mean).abs().max() <= bar
    assert (rd.cpu().double() - (0.9 * running.double() + 0.1 * mean)).abs().max() <= bar
    assert (y.cpu().double() - (x.double() - mean[chan][:, :, None])).abs().max() <= 2 * bar
