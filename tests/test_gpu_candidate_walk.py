"""Lists of marks at the sizes where they are handled differently: of at most 64 marks (walked as they are), of 65 to 128
(groups of one or two), of more than 2048 (handed over in parts), and rows that end inside a block of 256 or a slice of 512
inputs.  The table kernels, forced to run however many marks there are, against the kernels that evaluate every term: the
same bits, ties and positions included.  (Rows that are alike: tables per weight row; images against small weights: per batch row.)"""
import pytest
import torch

from test_gpu_candidate_random import _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1, 2, 3])
@pytest.mark.parametrize("B,CI,CO,K", [(1, 32, 1, 2), (129, 64, 127, 25), (3, 96, 130, 10), (127, 128, 3, 6), (65, 288, 70, 25),
                                       (300, 544, 33, 11), (130, 2048, 9, 10), (40, 2080, 129, 25), (140, 4640, 20, 3)])
def test_table_kernels_at_the_edges_of_their_lists(B, CI, CO, K, kind):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext, _lib
    dev = torch.device("cuda:0")
    import numpy as np
    g = torch.Generator().manual_seed(B + CI)
    x, w = _data(np.random.default_rng(CI), B, CI, CO, kind, g, dev)
    r = torch.rand(B, CI, 1, generator=g).to(dev) * 0.05
    xl, xu = (x - r).contiguous(), (x + r).contiguous()
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
                         lambda: ext.sort_neuron_forward(x, w, o[1], pk, 1, 0.75, K),
                         lambda: ext.bound_sort_neuron_forward(xl, xu, w, o[2], o[3], 1, 0.75, K),
                         lambda: ext.inf_dist_forward(x, w, o[4], p[0], 1),
                         lambda: ext.masked_inf_dist_forward(x, w, o[5], p[1], 1, 0.5, 7, ext.MASK_FACTORED),
                         lambda: ext.bound_inf_dist_forward_nograd(xl, xu, w, o[6], o[7], 1),
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
    if kind < 2 and CI >= 2048 and K <= 10:
        assert max(shares) < 1.0   # a table served every call
