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


@pytest.mark.parametrize("B,G,cnt,Cg,HW", [(40, 1, 6, 8, 1), (33, 2, 70, 70, 1), (600, 1, 100, 130, 1), (40, 1, 6, 8, 2)])
def test_lists_that_name_a_channel_more_than_once(B, G, cnt, Cg, HW):
    """One of the columns makes the channel's mean; all of them are shifted."""
    from sortnet_amd import ext
    g = torch.Generator().manual_seed(B)
    S = -(-B // 32)
    index = torch.randint(0, Cg, (S, G, cnt), generator=g).to(torch.int32)
    index[..., 1] = index[..., 0]
    x = torch.randn(B, G * cnt, HW, generator=g).cuda()
    chan = (index.long() + torch.arange(G)[None, :, None] * Cg).reshape(S, G * cnt).repeat_interleave(32, 0)[:B].cuda()
    y, mean = torch.full_like(x, float("nan")), torch.empty(G * Cg, device="cuda")
    ext.mean_shift_index_forward(x, index.cuda(), Cg, mean, None, 0.1, y)
    assert torch.equal(y, x - mean[chan][:, :, None])
