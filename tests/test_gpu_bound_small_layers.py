"""Interval bounds of the l-inf distance for layers between the smallest that are given tables per batch row and those given tables
per weight row too, with the built-in limits: odd numbers of rows and outputs, ties, undefined and infinite entries, inverted and
empty intervals, against the kernels that evaluate every term (the same bits, positions included)."""
import numpy as np
import pytest
import torch

from test_gpu_candidate_random import _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [0.02, 0.07, 1.0])   # tables serve, marks about the limit, every term
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
@pytest.mark.parametrize("B,CI,CO", [(513, 736, 751), (251, 3072, 1021), (1021, 1056, 327)])
def test_small_layers_with_tables_per_batch_row(B, CI, CO, kind, scale):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext, _lib
    dev = torch.device("cuda:0")
    assert 2 ** 27 + 3 * 2 ** 16 * CI <= B * CI * CO < 2 ** 31
    g = torch.Generator().manual_seed(B + CI)
    x, w = _data(np.random.default_rng(CI), B, CI, CO, kind, g, dev)
    w = (w * scale).contiguous()
    r = torch.rand(B, CI, 1, generator=g).to(dev) * 0.06 - 0.01
    xl, xu = (x - r).contiguous(), (x + r).contiguous()
    if kind == 3:
        xl[1, 5], xu[2, 7], xu[3, 40], xl[B - 1, CI - 1] = float("nan"), float("nan"), float("inf"), -float("inf")
        w[0, 9], w[CO - 1, 3] = float("nan"), float("inf")
    results = []
    try:
        for density in (0.0, -1.0):
            _lib.set_bound_candidate_density(density)
            o = [torch.full((B, CO, 1), float("nan"), device=dev) for _ in range(4)]
            p = [torch.full((B, CO, 1), -7, device=dev, dtype=torch.int32) for _ in range(2)]
            ext.bound_inf_dist_forward_nograd(xl, xu, w, o[0], o[1], 1)
            share = _lib.last_forward_term_share(torch.cuda.current_stream().cuda_stream)
            ext.bound_inf_dist_forward(xl, xu, w, o[2], o[3], p[0], p[1], 1)
            results.append(o + p)
    finally:
        _lib.set_bound_candidate_density(-1.0)
    if kind < 2 and scale == 0.02:
        assert share < 1.0
    for i, (a, b) in enumerate(zip(*results)):
        assert torch.equal(a, b), i
