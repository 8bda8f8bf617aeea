"""Candidate tables at the lengths of a row where their kernel changes: a wavefront alone, one to three blocks of 256 inputs per
wavefront (up to 4096, 8192 and 12288 inputs), rows that end inside a block, and longer ones, which are read twice; one to three
tiles of the other operand.  The table kernels, forced to run, against the kernels that evaluate every term: the same bits.  Rows
that are alike are served by the tables per weight row, images against small weights by those per batch row."""
import numpy as np
import pytest
import torch

from test_gpu_candidate_random import _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1, 3])
@pytest.mark.parametrize("CI", [32, 256, 288, 4064, 4096, 4128, 8192, 8224, 12288, 12320])
@pytest.mark.parametrize("B,CO", [(5, 130), (129, 3), (257, 258)])
def test_tables_of_rows_of_any_length(B, CI, CO, kind):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext, _lib
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(B + CI)
    x, w = _data(np.random.default_rng(CI), B, CI, CO, kind, g, dev)
    r = torch.rand(B, CI, 1, generator=g).to(dev) * 0.05 - 0.005   # some intervals are inverted
    xl, xu = (x - r).contiguous(), (x + r).contiguous()
    K = min(10, CI // 4)
    results, shares = [], []
    try:
        for density, form in ((0.0, 0), (1.0, 1), (1.0, 2)):
            _lib.set_sort_candidate_density(density)
            _lib.set_linf_candidate_density(density)
            _lib.set_bound_candidate_density(density)
            _lib.set_bound_candidate_form(form)
            o = [torch.full((B, CO, 1), float("nan"), device=dev) for _ in range(10)]
            p = [torch.full((B, CO, 1), -7, device=dev, dtype=torch.int32) for _ in range(4)]
            pk = torch.full((K, B, CO, 1), -7, device=dev, dtype=torch.int32)
            for call in (lambda: ext.sort_neuron_forward_nograd(x, w, o[0], 1, 0.75, K),
                         lambda: ext.bound_sort_neuron_forward(xl, xu, w, o[1], o[2], 1, 0.75, K),
                         lambda: ext.sort_neuron_forward(x, w, o[7], pk, 1, 0.75, K),
                         lambda: ext.inf_dist_forward(x, w, o[3], p[0], 1),
                         lambda: ext.masked_inf_dist_forward(x, w, o[4], p[1], 1, 0.5, 7, ext.MASK_FACTORED),
                         lambda: ext.bound_inf_dist_forward_nograd(xl, xu, w, o[5], o[6], 1),
                         lambda: ext.bound_inf_dist_forward(xl, xu, w, o[8], o[9], p[2], p[3], 1)):
                call()
                if density == 1.0 and (form == 1 or kind == 0):   # (the other form has no table per batch row)
                    shares.append(_lib.last_forward_term_share())
            results.append(o + p + [pk])
    finally:
        _lib.set_sort_candidate_density(-1.0)
        _lib.set_linf_candidate_density(-1.0)
        _lib.set_bound_candidate_density(-1.0)
        _lib.set_bound_candidate_form(0)
    for tables in results[1:]:
        for i, (a, b) in enumerate(zip(results[0], tables)):
            assert torch.equal(a, b), i
    if kind != 3 and CI >= 4064:
        assert max(shares) < 1.0   # a table served every call


@pytest.mark.parametrize("equal", [0, 2, 3, 40])   # ties of the K-th largest term: none, as many as are noted, one more, many
@pytest.mark.parametrize("B,CI,CO,K", [(130, 320, 9, 10), (128, 2144, 5, 2), (5, 4128, 3, 25)])
def test_positions_with_ties_of_the_smallest_entry(B, CI, CO, K, equal):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext, _lib
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(CI + equal)
    w = torch.randn(CO, CI, generator=g)
    x = torch.zeros(B, CI, 1)
    # row 0 holds K - 1 distinct large terms and 1 + equal terms of one value against every weight row
    for m in range(CO):
        at = torch.randperm(CI, generator=g)[:K + equal]
        w[m, at[:K - 1]] = 8 + torch.arange(K - 1) * 0.25
        w[m, at[K - 1:]] = -6.0
    x, w = x.to(dev), w.to(dev)
    results = []
    try:
        for density in (0.0, 1.0):
            _lib.set_sort_candidate_density(density)
            y = torch.full((B, CO, 1), float("nan"), device=dev)
            pos = torch.full((K, B, CO, 1), -7, device=dev, dtype=torch.int32)
            ext.sort_neuron_forward(x, w, y, pos, 1, 0.75, K)
            results.append((y, pos))
    finally:
        _lib.set_sort_candidate_density(-1.0)
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
