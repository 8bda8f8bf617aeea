"""Windows of a convolutional layer as columns and back, against torch's unfold and fold on the CPU."""
import pytest
import torch
import torch.nn.functional as TF

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape, kernel, dil, pad, stride", [
    ((1, 1, 1, 1), (1, 1), 1, 0, 1),          # one pixel
    ((3, 2, 7, 5), (3, 2), 1, 0, 1),          # ragged everything
    ((2, 3, 9, 11), (3, 3), 1, 1, 2),         # padding, stride
    ((2, 3, 12, 9), (3, 2), 2, 2, 3),         # dilation with a stride that skips taps
    ((5, 3, 32, 32), (30, 30), 1, 0, 2),      # the hybrid's first layer
    ((1, 4, 6, 6), (6, 6), 1, 0, 1),          # one position
])
def test_unfold_matches_torch(shape, kernel, dil, pad, stride):
    from sortnet_amd import ext
    g = torch.Generator().manual_seed(1)
    x = torch.randn(*shape, generator=g)
    xd = x.cuda().requires_grad_()
    y = ext.host().unfold(xd, *kernel, dil, pad, stride)
    ref = TF.unfold(x, kernel, dil, pad, stride)
    assert torch.equal(y.detach().cpu(), ref)
    gy = torch.randn(*ref.shape, generator=g)
    y.backward(gy.cuda())
    back = TF.fold(gy.double(), shape[2:], kernel, dil, pad, stride)
    # sums of at most kh * kw terms in fp32: each addition rounds to 2^-24 of a partial sum of unit-variance terms
    bound = 2.0 ** -23 * kernel[0] * kernel[1] * 5
    assert float((xd.grad.cpu().double() - back).abs().max()) <= bound


def test_unfold_refuses_a_window_that_does_not_fit():
    from sortnet_amd import ext
    with pytest.raises(RuntimeError, match="does not fit"):
        ext.host().unfold(torch.rand(1, 1, 4, 4, device="cuda"), 5, 5, 1, 0, 1)


@pytest.mark.parametrize("window", [1, 3])
def test_input_changed_in_place_between_the_passes(window):
    """The columns are the layer's own: what happens to the image after the forward does not concern the backward."""
    from sortnet_amd.layers import DropoutRegistry, NormDistConv
    layer = NormDistConv(3, 5, window, padding=window // 2, p=3.0, bias=False, mean_shift=False, registry=DropoutRegistry(1)).cuda()
    leaf = torch.rand(4, 3, 6, 6, generator=torch.Generator().manual_seed(2)).cuda().requires_grad_()
    want = torch.autograd.grad(layer(leaf)[0].sum(), [leaf, layer.weight])
    image = leaf * 1
    y = layer(image)[0]
    with torch.no_grad():
        image.mul_(2)
    for got, ref in zip(torch.autograd.grad(y.sum(), [leaf, layer.weight]), want):
        assert (got - ref).norm() <= 1e-5 * ref.norm()
    with torch.no_grad():
        assert torch.equal(layer(leaf)[0], y)
