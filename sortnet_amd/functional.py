"""Functional / autograd front-end of the distance-neuron kernels.

Public names, positional order, defaults, return shapes and dtypes follow the reference's
core/norm_dist.py (file:line cited per symbol) so that its layers (core/models/norm_dist.py)
run unmodified on top of this module.  Inputs are 3-D (B, C, HW) fp32 tensors on the GPU,
weight is (CO, CI / groups); outputs are fp32 on the input's device, positions are int32.

Every function dispatches to the HIP kernels through the native front-end (`ext.host()`, csrc/host.cpp).  `use_custom_cuda_func=False`
selects, as in the reference, a formulation in plain torch ops on the tensors' own device (differentiable
by autograd, formed for a bounded number of output channels at a time); it is a second, independent
statement of the same values and nothing in this library calls it on its own.
"""
import math

import torch

from . import ext as _C

__all__ = [
    "NormDistF", "NormDistDropoutF", "SortNeuronF", "BoundInfDistF", "MaskedInfDistF",
    "norm_dist", "norm_dist_dropout", "sort_neuron", "bound_sort_neuron", "bound_inf_dist", "masked_inf_dist",
    "MeanShiftF", "mean_shift", "MeanShiftIndexF", "mean_shift_index",
]


def _want_grad(*tensors):
    return torch.is_grad_enabled() and any(t.requires_grad for t in tensors)


# ---- use_custom_cuda_func=False: the reference's closed forms in torch ops ---------------------------------------
# The reference forms the whole (B, G, CO/G, CI/G, HW) tensor of differences at once (53.7 GB at B=512,
# CO=CI=5120); here the output channels go by in blocks whose differences stay below _TORCH_BLOCK_BYTES.
_TORCH_BLOCK_BYTES = 256 << 20


def _blocks_of_differences(inputs, weight, groups):
    """Yields, group by group and block by block of output channels, the differences
    d[k][b, m, n, hw] = inputs[k][b, g, n, hw] - weight[g, m, n] for every tensor of `inputs`, in the order in
    which the outputs are laid out ((B, G * CO/G, HW), group-major)."""
    B, C, HW = inputs[0].shape
    cig = C // groups
    cog = weight.size(0) // groups
    w = weight.view(groups, cog, cig)
    step = max(1, _TORCH_BLOCK_BYTES // max(1, 4 * len(inputs) * B * cig * HW))
    for g in range(groups):
        xs = [t[:, g * cig:(g + 1) * cig, :].unsqueeze(1) for t in inputs]        # (B, 1, cig, HW)
        for m0 in range(0, cog, step):
            wb = w[g, m0:m0 + step].unsqueeze(0).unsqueeze(-1)                    # (1, mc, cig, 1)
            yield [x - wb for x in xs]


def _torch_norm_dist(x, weight, p, groups):
    """core/norm_dist.py:181-185: the l-p norm of the differences, scaled by their largest magnitude (which is
    held constant under differentiation) so that large p neither overflows nor underflows."""
    out = []
    for (d,) in _blocks_of_differences([x], weight, groups):
        with torch.no_grad():
            scale = d.abs().amax(dim=2, keepdim=True)
        out.append((torch.linalg.vector_norm(d / scale, ord=p, dim=2, keepdim=True) * scale).squeeze(2))
    return torch.cat(out, dim=1)


def _torch_sort_neuron(x, weight, groups, q, truncate):
    """core/norm_dist.py:226-230: the `truncate` largest magnitudes, weighted q (1 - q)^j from the largest down and
    normalised by 1 - (1 - q)^truncate (no 1e-10 floor in this form)."""
    coef = ((1 - q) ** torch.arange(truncate, device=x.device, dtype=x.dtype) * q).view(1, 1, truncate, 1)
    out = []
    for (d,) in _blocks_of_differences([x], weight, groups):
        top = torch.topk(d.abs(), k=truncate, dim=2)[0]                            # (B, mc, truncate, HW), descending
        out.append((top * coef).sum(dim=2))
    return torch.cat(out, dim=1) / (1 - (1 - q) ** truncate)


def _torch_bound_inf_dist(x_lower, x_upper, weight, groups):
    """core/norm_dist.py:251-259: per input the two ends w - l and u - w; the upper result is the largest of their
    maxima and the lower result minus the smallest of their minima, both floored at 1e-10 (this form does not
    repair inverted intervals)."""
    lo, up = [], []
    for dl, du in _blocks_of_differences([x_lower, x_upper], weight, groups):
        t1, t2 = -dl, du
        up.append(torch.maximum(t1, t2).clamp(min=1e-10).amax(dim=2))
        lo.append((-torch.minimum(t1, t2).clamp(max=-1e-10)).amax(dim=2))
    return torch.cat(lo, dim=1), torch.cat(up, dim=1)


def _torch_norm_dist_dropout(x, weight, w_index_ci, w_index_co, p, groups):
    """core/norm_dist.py:195-213 without the kernels: each 32-sample sub-batch meets the sub-matrix of the weight
    that its two index lists select (a missing list keeps everything)."""
    cog, cig = weight.size(0) // groups, weight.size(1)
    w = weight.view(groups, cog, cig)
    out = []
    for s, b0 in enumerate(range(0, x.size(0), 32)):
        rows = []
        for g in range(groups):
            wg = w[g]
            if w_index_co is not None:
                wg = wg.index_select(0, w_index_co[s, g].long())
            if w_index_ci is not None:
                wg = wg.index_select(1, w_index_ci[s, g].long())
            rows.append(wg)
        out.append(_torch_norm_dist(x[b0:b0 + 32], torch.cat(rows, dim=0), p, groups))
    return torch.cat(out, dim=0)


# ---- the kernels' autograd ops -----------------------------------------------------------------------------------
# Forward, graph node and backward of every op are native (csrc/host.cpp); the classes below keep the reference's
# names and `apply` signatures.  `need_grad` and `tag` are accepted and not needed: positions are kept exactly when
# autograd records the call.
def _checked(x, weight, group):
    assert weight.size(1) * group == x.size(1)
    return _C.host()


def _check_power(p):
    if not (math.isinf(p) or p > 0):    # neither zero nor undefined
        raise NotImplementedError


class NormDistF:
    """l-p (finite p) or l-inf (p = inf) distance layer.  Mirrors core/norm_dist.py:6-51."""

    @staticmethod
    def apply(x, weight, group, p, need_grad=None, tag=None):
        host = _checked(x, weight, group)
        _check_power(p)
        return host.norm_dist(x, weight, group, p)


class NormDistDropoutF:
    """Distance layer on index-list sub-matrices of the weight, one list per 32-sample sub-batch.
    Mirrors core/norm_dist.py:54-99."""

    @staticmethod
    def apply(x, weight, w_index_ci, w_index_co, group, p, tag=None):
        assert weight.size(1) * group == x.size(1) or w_index_ci.size(-1) * group == x.size(1)
        _check_power(p)
        return _C.host().norm_dist_dropout(x, weight, w_index_ci, w_index_co, group, p)


class SortNeuronF:
    """Geometric-weighted sum of the top-`truncate` values of |x - w|.  Mirrors core/norm_dist.py:102-133."""

    @staticmethod
    def apply(x, weight, group, q, truncate, need_grad=None, tag=None):
        return _checked(x, weight, group).sort_neuron(x, weight, group, q, truncate)


class BoundInfDistF:
    """Interval bounds through the l-inf layer, forward and backward.  Mirrors core/norm_dist.py:136-173."""

    @staticmethod
    def apply(x_lower, x_upper, weight, group, need_grad=None, tag=None):
        assert x_lower.size() == x_upper.size()
        return _checked(x_lower, weight, group).bound_inf_dist(x_lower, x_upper, weight, group)


class MaskedInfDistF:
    """SortNet's training neuron as one fused op: max over a Bernoulli(q)-kept subset of |x - w|,
    the keep decisions drawn on the GPU from a stateless counter RNG of (seed, b, m, n).
    The reference builds the same kind of subset on the host (core/models/norm_dist.py:14-17) and
    feeds index lists to NormDistDropoutF; the backward here is the l-inf scatter through the
    saved arg-max index, identical to NormDistF's (core/norm_dist.py:29-39)."""

    @staticmethod
    def apply(x, weight, group, q, seed, mode, need_grad=None, tag=None):
        return _checked(x, weight, group).masked_inf_dist(x, weight, group, q, seed & 0xFFFFFFFF, mode)


class MeanShiftF:
    """y = x - mean_{b,hw}(x) with the mean inside the graph, plus the running-mean update the
    reference's MeanShiftDropout does under no_grad (core/models/bound_basic_module.py:123-157, the
    form without an index list).  The backward of the centring is the centring of the gradient."""

    @staticmethod
    def apply(x, running_mean, momentum):
        return _C.host().mean_shift(x, running_mean, momentum)


class MeanShiftIndexF:
    """MeanShiftF when every 32-sample sub-batch keeps its own channels (`index`, shape (S, G, cnt)):
    the mean of a channel runs over the sub-batches that kept it
    (core/models/bound_basic_module.py:125-137,146-153).  The backward is the same centring of the gradient."""

    @staticmethod
    def apply(x, index, channels, running_mean, momentum):
        if index is None:
            raise TypeError("mean_shift_index needs an index list; mean_shift is the form without one")
        return _C.host().mean_shift_index(x, index, channels, running_mean, momentum)


def mean_shift_index(x, index, channels, running_mean=None, momentum=0.1):
    """Training-mode mean shift of a compacted (B, G * cnt, HW) tensor; `channels` counts all channels of all
    groups.  Returns (x - mean[index], mean) and updates `running_mean` in place when given."""
    return MeanShiftIndexF.apply(x, index, channels, running_mean, momentum)


def mean_shift(x, running_mean=None, momentum=0.1):
    """Training-mode mean shift of a (B, C, HW) tensor; returns (x - mean, mean) and updates
    `running_mean` in place when given."""
    return MeanShiftF.apply(x, running_mean, momentum)


def norm_dist(input, weight, p, groups=1, use_custom_cuda_func=True, tag=None):
    """core/norm_dist.py:176-186."""
    if not use_custom_cuda_func:
        return _torch_norm_dist(input, weight, p, groups)
    return NormDistF.apply(input, weight, groups, p)


def norm_dist_dropout(input, weight, w_index_ci, w_index_co, p, groups=1, use_custom_cuda_func=True, tag=None):
    """core/norm_dist.py:191-214.  `input` is already compacted to the kept channels; `weight` is the
    full tensor; the same index list serves the 32 samples of a sub-batch."""
    if not use_custom_cuda_func:
        return _torch_norm_dist_dropout(input, weight, w_index_ci, w_index_co, p, groups)
    return NormDistDropoutF.apply(input, weight, w_index_ci, w_index_co, groups, p)


def sort_neuron(input, weight, groups=1, q=0.5, truncate=10, use_custom_cuda_func=True, tag=None):
    """core/norm_dist.py:217-231."""
    truncate = min(weight.size(-1), truncate)
    if q is None or q == 1.0 or truncate == 1:
        return norm_dist(input, weight, float("inf"), groups, tag=tag)
    if not use_custom_cuda_func:
        return _torch_sort_neuron(input, weight, groups, q, truncate)
    return SortNeuronF.apply(input, weight, groups, q, truncate)


def bound_sort_neuron(x_lower, x_upper, weight, groups=1, q=0.5, truncate=10, tag=None):
    """core/norm_dist.py:234-243.  Forward only, as in the reference."""
    truncate = min(weight.size(-1), truncate)
    if q is None or q == 1.0 or truncate == 1:
        return bound_inf_dist(x_lower, x_upper, weight, groups, tag=tag)
    assert not _want_grad(x_lower, x_upper, weight)
    return _C.host().bound_sort_neuron(x_lower, x_upper, weight, groups, q, truncate)


def bound_inf_dist(x_lower, x_upper, weight, groups=1, use_custom_cuda_func=True, tag=None):
    """core/norm_dist.py:246-260."""
    if not use_custom_cuda_func:
        return _torch_bound_inf_dist(x_lower, x_upper, weight, groups)
    return BoundInfDistF.apply(x_lower, x_upper, weight, groups)


# ---- evaluation pass: the values or bounds of a layer with sign * shift[channel] added, in one native call -----------------
# The same bits as the op above with the shift behind it; outside any graph.
def _kernels_can_add(vec, weight):
    """Whether the kernels take `vec` as it is (a call that torch would convert, broadcast or refuse is left to torch)."""
    return (vec.dtype == torch.float32 and vec.dim() == 1 and vec.size(0) == weight.size(0) and vec.device == weight.device
            and vec.is_contiguous() and vec.data_ptr() % 16 == 0)


def _shifted_values(x, weight, groups, q, shift, sign, truncate=10):
    truncate = min(weight.size(-1), truncate)
    host = _checked(x, weight, groups)
    if q is None or q == 1.0 or truncate == 1:
        return host.norm_dist_shifted(x, weight, groups, shift, sign)
    return host.sort_neuron_shifted(x, weight, groups, q, truncate, shift, sign)


def _shifted_bounds(x_lower, x_upper, weight, groups, q, shift, sign, truncate=10):
    truncate = min(weight.size(-1), truncate)
    assert x_lower.size() == x_upper.size()
    host = _checked(x_lower, weight, groups)
    if q is None or q == 1.0 or truncate == 1:
        return host.bound_inf_dist_shifted(x_lower, x_upper, weight, groups, shift, sign)
    return host.bound_sort_neuron_shifted(x_lower, x_upper, weight, groups, q, truncate, shift, sign)


def _shifted_box(x, x_lower, x_upper, weight, groups, q, shift, sign, truncate=10):
    """Values and bounds of one layer."""
    truncate = min(weight.size(-1), truncate)
    if q is None or q == 1.0 or truncate == 1 or x.size() != x_lower.size():
        return (_shifted_values(x, weight, groups, q, shift, sign, truncate),
                *_shifted_bounds(x_lower, x_upper, weight, groups, q, shift, sign, truncate))
    assert x_lower.size() == x_upper.size()
    return _checked(x, weight, groups).sort_neuron_box_shifted(x, x_lower, x_upper, weight, groups, q, truncate, shift, sign)


def masked_inf_dist(input, weight, q, seed, groups=1, mode=_C.MASK_TERM, tag=None):
    """Masked order-statistic neuron (see MaskedInfDistF).  `mode` is ext.MASK_TERM (independent
    draw per term) or ext.MASK_FACTORED (keep = keep_x(b, n) & keep_w(m, n))."""
    if q is None or q == 1.0:
        return norm_dist(input, weight, float("inf"), groups, tag=tag)
    return MaskedInfDistF.apply(input, weight, groups, q, seed, mode)
