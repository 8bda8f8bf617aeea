"""l-p distance at powers above 10, scale from a part of the inputs (layers of at least 2^29 terms): which outputs keep it, and what it may cost."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(x, w, p):
    d = (x[:, None, :].double() - w[None].double()).abs()
    top = d.amax(2)
    return (d / top[..., None]).pow(p).sum(2).pow(1 / p) * top


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


def test_error_where_the_part_misses_the_largest_differences():
    """Differences of about 1 in a column of the last chunk but one, the others 2^-11 of them. Relative to the largest difference an
    output has the roundings of the root (2 ulp at most: uniform, 6.9e-8 rms) and of the last product (3.4e-8), those of the logarithms
    near 0 count for nothing: 7.7e-8 rms. Exponents of 64 to 127 at p = 10.5 would add 2^-18 ln 2 / 10.5, 1.5e-7 rms; the line lies between."""
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(2)
    B, N, M = 64, 3200, 2640
    x, w = torch.randn(B, N, 1, generator=g, device="cuda") * 5e-5, torch.randn(M, N, generator=g, device="cuda") * 5e-5
    w[:, N - 40] = -1 - 0.03 * torch.rand(M, generator=g, device="cuda")
    y = F.norm_dist(x, w, 10.5)[..., 0]
    ref = torch.cat([_ref(x[b:b + 4, :, 0], w, 10.5) for b in range(0, B, 16)])
    err = torch.cat([y[b:b + 4] for b in range(0, B, 16)]).double() / ref - 1
    assert float(err.pow(2).mean().sqrt()) < 1.1e-7


def _us(fn, n=10):
    fn()
    times = []
    for _ in range(5):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(n):
            fn()
        e1.record()
        torch.cuda.synchronize()
        times.append(e0.elapsed_time(e1) * 1e3 / n)
    return min(times)


@pytest.mark.parametrize("B,N,M", [(1024, 1024, 8192), (2048, 1701, 4099)])
def test_part_is_taken_from_all_over_the_row(B, N, M):
    """Layers whose tiles fill the device without a split of the rows, three quarters of the inputs 100 times the others: a part from all over the row holds some of them, one from its start does not, and the
    layer runs both steps twice (1.8 times as long). A quarter more is the limit."""
    from sortnet_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = torch.randn(B, N, 1, generator=g, device="cuda") * 0.3, torch.randn(M, N, generator=g, device="cuda")
    ci = torch.arange(0, N, dtype=torch.int32, device="cuda").expand(B // 32, 1, N).contiguous()
    even = _us(lambda: F.norm_dist_dropout(x, w, ci, None, 24.0))
    w[:, N // 4:] *= 100
    x[:, N // 4:] *= 100
    assert _us(lambda: F.norm_dist_dropout(x, w, ci, None, 24.0)) < 1.25 * even
