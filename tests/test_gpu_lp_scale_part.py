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


@pytest.mark.parametrize("B,N,M,lists", [(64, 10240, 1024, False), (96, 3001, 2513, True), (250, 3072, 1021, False), (512, 2048, 1024, False)])
def test_outputs_do_not_depend_on_the_batch(B, N, M, lists):
    """A sample whose differences are far above the others' is formed from all inputs; the outputs of the others keep their bits."""
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = torch.randn(B, N, 1, generator=g, device="cuda") * 0.3, torch.randn(M, N + 99 * lists, generator=g, device="cuda")
    ci = torch.arange(0, N, dtype=torch.int32, device="cuda").expand(B // 32, 1, N).contiguous() if lists else None

    def y():
        return (F.norm_dist_dropout(x, w, ci, None, 24.0) if lists else F.norm_dist(x, w, 24.0))[..., 0]
    before = y()
    other = torch.arange(B, device="cuda") != 5
    kept = x[5].clone()
    x[5, N - 40] = 3e4
    assert torch.equal(y()[other], before[other])
    assert ((y()[5] - 3e4).abs() < 10).all()
    x[5] = kept
    x[5, N - 40] = float("nan")
    assert torch.equal(y()[other], before[other]) and y()[5].isnan().all()
    x[5] = kept
    keep = torch.arange(M, device="cuda") != 7
    w[7, N - 40] = 1e4
    assert torch.equal(y()[:, keep], before[:, keep])
