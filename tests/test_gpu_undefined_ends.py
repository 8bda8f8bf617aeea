"""Intervals with one undefined end: each result takes the term of the defined end (core/cuda/sort_neuron.cu:262-290,
core/cuda/bound_inf_dist_cuda.cu:63-90), so the upper result of such an input may be below its lower one.  Tables per batch row,
forced to run, against the kernels that evaluate every term: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,CI,CO,K", [(70, 512, 150, 5), (9, 4128, 40, 10), (130, 8224, 9, 2), (5, 12320, 130, 25)])
def test_bounds_with_one_undefined_end(B, CI, CO, K):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext, _lib
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(CI)
    x = torch.rand(B, CI, 1, generator=g)
    w = (torch.randn(CO, CI, generator=g) * CI ** -0.5).to(dev)
    r = torch.rand(B, CI, 1, generator=g) * 0.03
    xl, xu = x - r, x + r
    nan = float("nan")
    at = torch.randperm(CI, generator=g)[:8 * K]
    for i, n in enumerate(at.tolist()):
        xl[0, n], xu[0, n] = nan, -5.0 - i / 64          # every third row: lower ends, upper ends, both
        xl[1, n], xu[1, n] = 6.0 + i / 64, nan
        xl[2, n], xu[2, n] = (nan, -4.0 - i / 64) if i % 2 else (nan, nan)
    for t in (xl, xu):
        t[3:] = t[torch.arange(3, B) % 3]
    xl, xu = xl.contiguous().to(dev), xu.contiguous().to(dev)
    results = []
    try:
        for density in (0.0, 1.0):
            _lib.set_sort_candidate_density(density)
            _lib.set_bound_candidate_density(density)
            o = [torch.full((B, CO, 1), nan, device=dev) for _ in range(4)]
            p = [torch.full((B, CO, 1), -7, device=dev, dtype=torch.int32) for _ in range(2)]
            ext.bound_sort_neuron_forward(xl, xu, w, o[0], o[1], 1, 0.75, K)
            share = _lib.last_forward_term_share()
            ext.bound_inf_dist_forward(xl, xu, w, o[2], o[3], p[0], p[1], 1)
            results.append(o + p)
    finally:
        _lib.set_sort_candidate_density(-1.0)
        _lib.set_bound_candidate_density(-1.0)
    assert share < 1.0   # the tables served
    for i, (a, b) in enumerate(zip(*results)):
        assert torch.equal(a, b), i
