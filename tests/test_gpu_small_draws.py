"""Kept-channel lists are the same whichever stream draws them, an empty one among them, and a layer's draw goes to the second
stream by the layer's work."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sub_batches,groups,channels,q", [(1, 1, 256, 0.75), (8, 1, 4095, 0.5), (8, 1, 4096, 0.5), (3, 2, 100, 0.3),
                                                           (2, 1, 17, 0.0)])
def test_lists_do_not_depend_on_the_stream(sub_batches, groups, channels, q):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext
    from sortnet_amd.layers import DropoutRegistry
    reg = DropoutRegistry(5)
    for draw in range(1, 5):
        lists = reg.sample(sub_batches, groups, channels, q, torch.device("cuda:0"), host_paced=draw % 2 == 0)
        seed = (5 * 1000003 + draw) & 0xFFFFFFFF
        ref = ext.sample_index_lists(seed, sub_batches, groups, channels, ext.mask_count(seed, channels, q), torch.device("cuda:0"))
        assert lists.dtype == torch.int32 and lists.shape == ref.shape and torch.equal(lists, ref)


# few samples, wide: the draw is small (8192 and fewer channels), the layer is not
@pytest.mark.parametrize("batch,width,p,second", [(32, 5120, 24.0, True), (32, 256, 24.0, False), (32, 5120, 8.0, True),
                                                  (64, 2048, 8.0, False), (64, 1536, math.inf, False)])
def test_draws_of_large_layers_overlap(batch, width, p, second):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd.layers import DropoutRegistry, NormDist
    reg = DropoutRegistry(3)
    with torch.device("cuda"):
        layers = [NormDist(width, width, bias=False, p=p, dropout=d, registry=reg) for d in (1.0, 0.75)]
    paced = []
    sample = reg.sample
    reg.sample = lambda *a, **k: (paced.append(a[5] if len(a) > 5 else k.get("host_paced", False)), sample(*a, **k))[1]
    layers[0].train()(torch.rand(batch, width, device="cuda"))
    assert paced == [not second] and (len(reg._side_streams) == 1) == second
