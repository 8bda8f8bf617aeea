"""Gradient of the sort neuron to its input (core/cuda/sort_neuron.cu:196-240): from 512 inputs on, where a layer has few rows,
several workgroups share a row, each with a part of the inputs.  Parts of equal and unequal length, two to eight of them, groups,
several positions per row, and counts of terms around the five that are in flight, against the CPU oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,q", [(2, 0.75), (5, 0.3), (7, 1.0), (25, 0.3)])
@pytest.mark.parametrize("B,CI,CO,G,HW", [(3, 511, 70, 1, 1),       # one part still
                                          (3, 512, 70, 1, 1), (300, 517, 20, 1, 1),    # two
                                          (5, 2062, 66, 2, 3),      # four of 1031 inputs, groups and positions
                                          (2, 2307, 40, 1, 1), (1, 12287, 129, 1, 1)])  # eight
def test_input_gradient_in_parts(oracle, B, CI, CO, G, HW, K, q):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sortnet_amd import ext
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(CI + K)
    n = CI // G
    ends = np.array([n * i // 8 + d for i in range(9) for d in (-1, 0)])
    ends = ends[(ends >= 0) & (ends < n)]         # first and last inputs of every part
    pos = rng.integers(0, n, (K, B, CO, HW))
    pos = np.where(rng.random(pos.shape) < 0.3, rng.choice(ends, pos.shape), pos).astype(np.uint32)
    pos = (pos | (rng.integers(0, 2, pos.shape).astype(np.uint32) << 31)).view(np.int32)
    gy = rng.standard_normal((B, CO, HW)).astype(np.float32)
    ref, ref_w = oracle.sort_neuron_backward(gy, pos, (B, CI, HW), (CO, n), q, K, G)
    gd, pd = torch.from_numpy(gy).to(dev), torch.from_numpy(pos).to(dev)
    gx, gx2 = (torch.full((B, CI, HW), float("nan"), device=dev) for _ in range(2))
    gw = torch.full((CO, n), float("nan"), device=dev)
    ext.sort_neuron_backward_input(gd, pd, gx, G, q, K)
    ext.sort_neuron_backward_input_weight(gd, pd, gx2, gw, G, q, K)
    # an input is sent at most CO * K values, most of them far fewer: sums in any order agree to 1e-5 of the largest
    for got, want in ((gx, ref), (gx2, ref), (gw, ref_w)):
        np.testing.assert_allclose(got.cpu().numpy(), want, rtol=1e-5, atol=1e-5 * float(np.abs(want).max()))
