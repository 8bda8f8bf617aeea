"""Arguments that the front-end refuses before any device work: an exception, never an abort or a launch."""
import math

import pytest
import torch

from sortnet_amd import ext
from sortnet_amd import functional as F

X, W = torch.ones(2, 3, 1), torch.ones(4, 3)


@pytest.mark.parametrize("p", [0.0, -2.0, math.nan])
def test_powers_without_a_meaning(p):
    with pytest.raises(NotImplementedError):
        F.norm_dist(X, W, p)
    with pytest.raises(NotImplementedError):
        F.norm_dist_dropout(X, W, None, None, p)


@pytest.mark.parametrize("call", [
    lambda: F.norm_dist(X, W, 2.0), lambda: F.norm_dist(X, W, math.inf), lambda: F.norm_dist(X, W, -math.inf),
    lambda: F.norm_dist_dropout(X, W, None, None, 8.0), lambda: F.sort_neuron(X, W, q=0.5, truncate=2),
    lambda: F.bound_inf_dist(X, X, W), lambda: F.bound_sort_neuron(X, X, W, q=0.5, truncate=2), lambda: F.masked_inf_dist(X, W, 0.5, -3),
    lambda: F.mean_shift(X), lambda: F.mean_shift_index(X, torch.zeros(1, 1, 3, dtype=torch.int32), 4),
    lambda: ext.host().channel_shift(X, torch.ones(3), 1.0), lambda: ext.host().unfold(torch.ones(1, 1, 4, 4), 2, 2, 1, 0, 1)])
def test_tensors_on_the_host(call):
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        call()


def test_missing_dimensions():
    for call in (lambda: F.norm_dist(X[..., 0], W, 2.0), lambda: F.sort_neuron(X[..., 0], W, q=0.5, truncate=2),
                 lambda: F.bound_inf_dist(X[..., 0], X[..., 0], W), lambda: F.mean_shift(X[..., 0]), lambda: ext.host().unfold(X, 1, 1, 1, 0, 1)):
        with pytest.raises((IndexError, RuntimeError)):
            call()


def test_lists_without_groups_and_windows_without_steps():
    with pytest.raises(TypeError):
        F.mean_shift_index(X, None, 4)
    with pytest.raises(RuntimeError, match="groups"):
        F.mean_shift_index(X, torch.zeros(1, 0, 3, dtype=torch.int32), 4)
    for stride in (0, -1):
        with pytest.raises(RuntimeError, match="stride"):
            ext.host().unfold(torch.ones(1, 1, 4, 4), 2, 2, 1, 0, stride)
