"""Sort neuron: up to which marked share the tables per weight row serve the values, with the built-in limit.  Rows of fewer than 320
inputs stop at a tenth, since the kernels that form every term are done sooner there."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,CI,CO,spread,serves", [(512, 256, 256, 0.6, False), (512, 288, 260, 0.6, False), (512, 256, 256, 0.1, True),
                                                   (100, 480, 450, 0.6, True), (300, 320, 256, 0.6, True)])
def test_short_rows_have_a_lower_limit(B, CI, CO, spread, serves):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext, _lib
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(CI + CO)
    x = (torch.randn(1, CI, 1, generator=g) * 0.3 + torch.randn(B, CI, 1, generator=g) * 0.3 * spread).to(dev)
    w = torch.randn(CO, CI, generator=g).to(dev)
    y = torch.empty(B, CO, 1, device=dev)

    def share():
        ext.sort_neuron_forward_nograd(x, w, y, 1, 0.3, 10)
        return _lib.last_forward_term_share()
    try:
        _lib.set_sort_candidate_density(1.0)
        marked = share()
    finally:
        _lib.set_sort_candidate_density(-1.0)
    assert 0.12 < marked < 0.38 if spread > 0.5 else 0.01 < marked < 0.10
    assert share() == (marked if serves else 1.0)
