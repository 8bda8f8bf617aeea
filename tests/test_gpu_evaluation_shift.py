"""Evaluation pass: the mean shift or bias behind a layer, added by the kernels that store its values, has the bits of the two steps
one after the other - whichever kernel serves the layer - and steps that have to be seen to run still do."""
import pytest
import torch

from sortnet_amd import _lib, ext
from sortnet_amd import functional as F
from sortnet_amd.ell_inf_models import SortMLPModel
from sortnet_amd.layers import DropoutRegistry, MeanShiftDropout, NormDist
from sortnet_amd.model import DistanceMLP

pytestmark = pytest.mark.gpu


def _plus(y, shift, sign):
    return y + sign * shift.view(1, -1, 1)


# rows x inputs x outputs: streamed weights (few rows, ragged, long), every term (one and two levels, narrow and wide), tables per
# weight row (spread 0.3) and per batch row (images against small weights), padded copies
SHAPES = [(1, 640, 513), (3, 31, 7), (40, 1999, 300), (64, 2048, 2048), (130, 250, 257), (512, 100, 36), (128, 1306, 1306),
          (128, 3072, 1024), (257, 1024, 1030)]


@pytest.mark.parametrize("density", [-1.0, 0.0, 1.0])
@pytest.mark.parametrize("images", [False, True])
@pytest.mark.parametrize("B,N,M", SHAPES)
def test_same_bits_as_two_steps(B, N, M, images, density):
    g = torch.Generator(device="cuda").manual_seed(B + N + M)
    x = torch.rand(B, N, 1, device="cuda", generator=g)
    w = torch.randn(M, N, device="cuda", generator=g)
    if images:
        w.mul_(N ** -0.5)
    else:
        x = (x - 0.5) * 0.3
    lo, up = x - 0.02, x + 0.02
    shift = torch.randn(M, device="cuda", generator=g)
    _lib.set_sort_candidate_density(density)
    _lib.set_linf_candidate_density(density)
    _lib.set_bound_candidate_density(density)
    try:
        for q in (0.75, None):
            for sign in (1.0, -1.0):
                assert torch.equal(F._shifted_values(x, w, 1, q, shift, sign), _plus(F.sort_neuron(x, w, q=q), shift, sign))
                for got, want in zip(F._shifted_bounds(lo, up, w, 1, q, shift, sign), F.bound_sort_neuron(lo, up, w, q=q)):
                    assert torch.equal(got, _plus(want, shift, sign))
    finally:
        _lib.set_sort_candidate_density(-1.0)
        _lib.set_linf_candidate_density(-1.0)
        _lib.set_bound_candidate_density(-1.0)


@pytest.mark.parametrize("groups,HW", [(2, 1), (1, 5), (3, 4)])
def test_groups_and_positions(groups, HW):
    g = torch.Generator(device="cuda").manual_seed(groups + HW)
    x = torch.randn(33, 36 * groups, HW, device="cuda", generator=g)
    w = torch.randn(17 * groups, 36, device="cuda", generator=g)
    shift = torch.randn(17 * groups, device="cuda", generator=g)
    for q in (0.5, None):
        assert torch.equal(F._shifted_values(x, w, groups, q, shift, -1.0), _plus(F.sort_neuron(x, w, groups, q=q), shift, -1.0))
        for got, want in zip(F._shifted_bounds(x, x + 0.1, w, groups, q, shift, -1.0), F.bound_sort_neuron(x, x + 0.1, w, groups, q=q)):
            assert torch.equal(got, _plus(want, shift, -1.0))


def _layer_by_layer(model, x, eps):
    """The pass of SortMLPModel with the shift behind every layer as a step of its own."""
    paras = [z.reshape(z.size(0), -1, 1) for z in (x, (x - eps).clamp(min=0), (x + eps).clamp(max=1))]
    for layer in model.fc_dist:
        y = F.sort_neuron(paras[0], layer.weight, q=layer.dropout)
        lo, up = F.bound_sort_neuron(paras[1], paras[2], layer.weight, q=layer.dropout)
        vec, sign = (layer.mean_shift.running_mean, -1.0) if layer.mean_shift is not None else (layer.bias, 1.0)
        paras = [_plus(z, vec, sign) for z in (y, lo, up)]
    return [z.squeeze(-1) for z in paras]


@pytest.mark.parametrize("batch", [1, 48])
def test_models(batch):
    torch.manual_seed(3)
    model = SortMLPModel(4, 256, (1, 28, 28), dropout=0.75, std=1.0, registry=DropoutRegistry(1)).cuda().eval()
    for m in model.modules():
        if isinstance(m, MeanShiftDropout):
            m.running_mean.normal_()
    model.fc_dist[-1].bias.data.normal_()
    x = torch.rand(batch, 1, 28, 28, device="cuda")
    with torch.no_grad():
        want = _layer_by_layer(model, x, 0.03)
        zero, one = torch.zeros((), device="cuda"), torch.ones((), device="cuda")
        flat = [z.reshape(batch, -1) for z in (x, torch.maximum(x - 0.03, zero), torch.minimum(x + 0.03, one))]
        for got, ref in zip(model.fc_dist(flat), want):
            assert torch.equal(got, ref)
        assert torch.equal(model(x), -want[0])
    assert torch.equal(model(x).detach(), -want[0])          # with a graph: the shift is a step of its own
    net = DistanceMLP(784, 300, 3, 10, q=None)
    for m in net.running_mean:
        m.normal_()
    net.bias.data.normal_()
    h = x.reshape(batch, -1, 1)
    lo, up = h - 0.03, h + 0.03
    for i, w in enumerate(net.weights):
        vec, sign = (net.running_mean[i], -1.0) if i < 2 else (net.bias, 1.0)
        with torch.no_grad():
            h = _plus(F.norm_dist(h, w, float("inf")), vec, sign)
            lo, up = [_plus(z, vec, sign) for z in F.bound_inf_dist(lo, up, w)]
    first = x.reshape(batch, -1)
    assert torch.equal(net.predict(first), h.squeeze(-1))
    for got, ref in zip(net.bounds(first - 0.03, first + 0.03), (lo, up)):
        assert torch.equal(got, ref.squeeze(-1))


class _Doubled(MeanShiftDropout):
    def forward(self, x=None, lower=None, upper=None, index=None):
        return tuple(None if z is None else 2 * z for z in (x, lower, upper))


def test_steps_that_have_to_be_seen():
    layer = NormDist(64, 40, bias=True, registry=DropoutRegistry(0)).cuda().eval()
    layer.mean_shift.running_mean.normal_()
    layer.bias.data.normal_()
    x = torch.randn(5, 64, device="cuda")
    y = F.norm_dist(x.unsqueeze(-1), layer.weight, float("inf")).detach().squeeze(-1)
    with torch.no_grad():
        want = (y - layer.mean_shift.running_mean) + layer.bias
        assert torch.equal(layer(x)[0], want)
        seen = []
        handle = layer.mean_shift.register_forward_hook(lambda m, a, out: seen.append(1))
        assert torch.equal(layer(x)[0], want) and seen == [1]
        handle.remove()
        layer.mean_shift.__class__ = _Doubled
        assert torch.equal(layer(x)[0], 2 * y + layer.bias)
        layer.mean_shift.__class__ = MeanShiftDropout
        # a mean that the kernels do not take as it is goes through the step itself, which refuses it
        layer.mean_shift.running_mean = torch.randn(41, device="cuda")[1:]
        with pytest.raises(RuntimeError, match="aligned"):
            layer(x)
        layer.mean_shift.running_mean = torch.randn(40, device="cuda", dtype=torch.float64)
        with pytest.raises(RuntimeError, match="dtype"):
            layer(x)
    plain = NormDist(64, 40, bias=True, mean_shift=False, registry=DropoutRegistry(0)).cuda().eval()
    plain.bias.data = torch.randn(40, device="cuda", dtype=torch.float64)
    with torch.no_grad():
        out = plain(x)[0]
    assert out.dtype == torch.float64


def test_arguments_are_checked():
    x, w = torch.randn(4, 32, 1, device="cuda"), torch.randn(8, 32, device="cuda")
    shift = torch.randn(8, device="cuda")
    with pytest.raises(RuntimeError, match="sign"):
        ext.host().sort_neuron_shifted(x, w, 1, 0.5, 10, shift, 0.5)
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        ext.host().norm_dist_shifted(x, w, 1, shift.cpu(), 1.0)


# one table for values and bounds: served (whole and padded rows, tiles that are not full), too many marks for the bounds alone (wide
# intervals), undefined and infinite entries, inputs outside their intervals, intervals turned round
@pytest.mark.parametrize("density", [-1.0, 0.03, 1.0])
@pytest.mark.parametrize("width", [0.02, 3.0])
@pytest.mark.parametrize("B,N,M", [(128, 320, 450), (257, 1024, 300), (200, 1306, 700), (130, 4443, 515), (384, 5120, 129), (150, 12320, 64)])
def test_box_has_the_bits_of_both_calls(B, N, M, width, density):
    g = torch.Generator(device="cuda").manual_seed(B + N)
    x = torch.randn(B, N, 1, device="cuda", generator=g).mul_(0.1)
    w = torch.randn(M, N, device="cuda", generator=g)
    lo, up = x - width, x + width
    lo[3, 5], up[3, 5] = up[3, 5].clone(), lo[3, 5].clone()
    x[1, 7] = 9.0
    x[2, 3], lo[4, 1], up[5, 2], w[6, 4], w[7, 8] = float("nan"), float("-inf"), float("inf"), float("inf"), float("nan")
    shift = torch.randn(M, device="cuda", generator=g)
    _lib.set_sort_candidate_density(density)
    try:
        want = [F._shifted_values(x, w, 1, 0.75, shift, -1.0), *F._shifted_bounds(lo, up, w, 1, 0.75, shift, -1.0)]
        for _ in range(6):                                    # as the hints learn
            for got, ref in zip(F._shifted_box(x, lo, up, w, 1, 0.75, shift, -1.0), want):
                assert torch.equal(got.nan_to_num(nan=-1.0), ref.nan_to_num(nan=-1.0))
            torch.cuda.synchronize()
    finally:
        _lib.set_sort_candidate_density(-1.0)


def test_box_under_capture():
    """Recorded before and after a call has sized the workspace, replayed on narrow and wide intervals."""
    g = torch.Generator(device="cuda").manual_seed(11)
    B, N, M = 256, 1024, 512
    w = torch.randn(M, N, device="cuda", generator=g)
    shift = torch.randn(M, device="cuda", generator=g)
    x = torch.randn(B, N, 1, device="cuda", generator=g).mul_(0.1)
    lo, up = x - 0.02, x + 0.02
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(3):
            F._shifted_box(x, lo, up, w, 1, 0.75, shift, -1.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = F._shifted_box(x, lo, up, w, 1, 0.75, shift, -1.0)
    for width in (0.02, 2.0, 0.0, 5.0, 0.02):
        x.copy_(torch.randn(B, N, 1, device="cuda", generator=g).mul_(0.1))
        lo.copy_(x - width)
        up.copy_(x + width)
        graph.replay()
        torch.cuda.synchronize()
        want = [F._shifted_values(x, w, 1, 0.75, shift, -1.0), *F._shifted_bounds(lo, up, w, 1, 0.75, shift, -1.0)]
        for got, ref in zip(out, want):
            assert torch.equal(got, ref)
