"""l-p distance at powers above 10, scale from a part of the inputs (layers of at least 2^29 terms): which outputs keep it, and what it may cost."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,M", [(64, 3200, 2622), (32, 320, 262)])
@pytest.mark.parametrize("at", [7, -1])
def test_differences_near_the_largest_number(B, N, M, at):
    """Largest differences above 2^126, whose reciprocal is subnormal: the layer's other terms vanish beside them, so the result is the difference
    itself, to the 2 ulp of the root, the rounding of the power's scale (log2 of 128, an ulp each of it and of the difference's) and the product's."""
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = torch.randn(B, N, 1, generator=g, device="cuda") * 0.3, torch.randn(M, N, generator=g, device="cuda")
    far = {3: 1.0e38, M // 2: 1.9e38, M - 1: -3.2e38}
    for m, v in far.items():
        w[m, at] = v
    y = F.norm_dist(x, w, 24.0)[..., 0]
    for m, v in far.items():
        assert ((y[:, m].double() - abs(v)).abs() <= (2 ** -15 + 2 ** -22) * abs(v)).all(), (m, y[:, m])
    assert torch.isfinite(y).all()
