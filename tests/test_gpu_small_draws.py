"""Kept-channel lists are the same whichever stream draws them: layers on either side of the size from which the draw goes to
a second stream, and an empty list."""
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
    for draw in range(1, 4):
        lists = reg.sample(sub_batches, groups, channels, q, torch.device("cuda:0"))
        seed = (5 * 1000003 + draw) & 0xFFFFFFFF
        ref = ext.sample_index_lists(seed, sub_batches, groups, channels, ext.mask_count(seed, channels, q), torch.device("cuda:0"))
        assert lists.dtype == torch.int32 and lists.shape == ref.shape and torch.equal(lists, ref)
