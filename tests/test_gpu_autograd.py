"""Graph nodes of the native front-end: gradients with respect to any subset of the inputs, and what the nodes refuse."""
import itertools
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _op(name):
    """(inputs, function of them): the inputs are leaves that require gradients, the function returns the outputs that
    gradients flow from."""
    from sortnet_amd import ext
    from sortnet_amd import functional as F
    g = torch.Generator().manual_seed(5)
    B, n, m = 70, 96, 40
    x, w = torch.randn(B, n, 1, generator=g).cuda(), torch.randn(m, n, generator=g).cuda()
    if name.startswith("norm_dist "):
        p = float(name.split()[1])
        return [x, w], lambda x, w: [F.norm_dist(x, w, p)]
    if name.startswith("lists "):
        p = float(name.split()[1])
        keep = lambda c, k: torch.rand(3, 1, c, generator=g).argsort(-1)[..., :k].sort(-1)[0].to(torch.int32).cuda()   # noqa: E731
        ci, co = keep(n, 64), keep(m, 30)
        return [x[:, :64].contiguous(), w], lambda x, w: [F.norm_dist_dropout(x, w, ci, co, p)]
    if name == "sort_neuron":
        return [x, w], lambda x, w: [F.sort_neuron(x, w, q=0.6)]
    if name == "masked_inf_dist":
        return [x, w], lambda x, w: [F.masked_inf_dist(x, w, 0.5, 3)]
    if name == "bound_inf_dist":
        return [x - 0.1, x + 0.1, w], lambda l, u, w: list(F.bound_inf_dist(l, u, w))
    if name == "mean_shift":
        return [x], lambda x: [F.mean_shift(x)[0]]
    if name == "mean_shift_index":
        index = torch.rand(3, 1, 130, generator=g).argsort(-1)[..., :n].to(torch.int32).cuda()
        return [x], lambda x: [F.mean_shift_index(x, index, 130)[0]]
    assert name == "unfold"
    return [torch.randn(5, 3, 9, 7, generator=g).cuda()], lambda x: [ext.host().unfold(x, 3, 2, 1, 1, 2)]


OPS = ["norm_dist inf", "norm_dist 3", "norm_dist 24", "lists inf", "lists 8", "sort_neuron", "masked_inf_dist", "bound_inf_dist",
       "mean_shift", "mean_shift_index", "unfold"]


def _graph(name):
    inputs, fn = _op(name)
    inputs = [t.requires_grad_() for t in inputs]
    outs = fn(*inputs)
    g = torch.Generator().manual_seed(6)
    return inputs, outs, [torch.randn(o.shape, generator=g).cuda() for o in outs]


def _close(a, b):
    # the same addends in another order (gradients merge by fp32 additions in memory)
    assert a.shape == b.shape and (a - b).norm() <= 1e-5 * b.norm()


@pytest.mark.parametrize("name", OPS)
def test_gradients_of_any_subset_of_the_inputs(name):
    inputs, outs, gys = _graph(name)
    torch.autograd.backward(outs, gys, retain_graph=True)
    full = [t.grad for t in inputs]
    assert all(t is not None and t.norm() > 0 for t in full)
    for k in range(1, len(inputs) + 1):
        for subset in itertools.combinations(range(len(inputs)), k):
            got = torch.autograd.grad(outs, [inputs[i] for i in subset], gys, retain_graph=True)
            for i, t in zip(subset, got):
                _close(t, full[i])


@pytest.mark.parametrize("wanted", [w for w in itertools.product([False, True], repeat=3) if any(w)])
def test_bound_gradients_by_what_requires_them(wanted):
    """One bound alone, with a frozen weight, gets zeros (core/norm_dist.py:157-173); every other set gets its gradients, also
    when only a part of it is asked for."""
    from sortnet_amd import functional as F
    inputs, outs, gys = _graph("bound_inf_dist")
    full = torch.autograd.grad(outs, inputs, gys)
    some = [t.detach().clone().requires_grad_(r) for t, r in zip(inputs, wanted)]
    outs = F.bound_inf_dist(*some)
    for i, t in enumerate(some):
        if wanted[i]:
            got, = torch.autograd.grad(outs, [t], gys, retain_graph=True)
            if sum(wanted) == 1 and not wanted[2]:
                assert got.shape == t.shape and not got.any()
            else:
                _close(got, full[i])


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("name", OPS)
def test_forward_mode_is_refused(name, grad):
    """There is no forward-mode formula: an output without a tangent would pass for a zero derivative."""
    import torch.autograd.forward_ad as fw
    inputs, fn = _op(name)
    for i in range(len(inputs)):
        with fw.dual_level(), torch.set_grad_enabled(grad):
            dual = [fw.make_dual(t, torch.ones_like(t)) if j == i else t for j, t in enumerate(inputs)]
            with pytest.raises(NotImplementedError, match="forward mode"):
                fn(*dual)


@pytest.mark.parametrize("name", OPS)
def test_function_transforms_are_refused(name):
    inputs, fn = _op(name)
    with pytest.raises(RuntimeError, match="torch.func"):
        torch.func.grad(lambda t: fn(t, *inputs[1:])[0].sum())(inputs[0])
    with pytest.raises(RuntimeError, match="torch.func"):
        torch.func.vmap(lambda s: fn(*inputs)[0].sum() * s)(torch.ones(2, device="cuda"))


def _run(threads):
    for t in threads:
        t.start()
    for t in threads:
        t.join()


@pytest.mark.parametrize("name", OPS)
def test_two_threads_run_backward_through_one_graph(name):
    inputs, outs, gys = _graph(name)
    full = torch.autograd.grad(outs, inputs, gys, retain_graph=True)
    wrong = []

    def retained():
        for _ in range(20):
            for a, b in zip(torch.autograd.grad(outs, inputs, gys, retain_graph=True), full):
                if not (a - b).norm() <= 1e-5 * b.norm():
                    wrong.append(name)

    _run([threading.Thread(target=retained) for _ in range(2)])
    assert not wrong

    def released():                     # frees what the nodes saved: the other pass gets its gradients or is told so
        try:
            got = torch.autograd.grad(outs, inputs, gys)
        except RuntimeError as e:
            if "second time" not in str(e):
                wrong.append(str(e))
            return
        for a, b in zip(got, full):
            if not (a - b).norm() <= 1e-5 * b.norm():
                wrong.append(name)

    _run([threading.Thread(target=released) for _ in range(2)])
    assert not wrong


@pytest.mark.parametrize("name", OPS)
def test_saved_tensor_hooks_and_second_pass(name):
    inputs, outs, gys = _graph(name)
    full = torch.autograd.grad(outs, inputs, gys)
    if name not in ("mean_shift", "unfold"):        # these save nothing
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(outs, inputs, gys)
    recorded = []

    def unpack(packed):                 # runs with autograd as the caller left it
        if packed.is_floating_point() and torch.is_grad_enabled():
            leaf = packed.detach().requires_grad_()
            recorded.append((leaf * 2).requires_grad)
        return packed.cuda()

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), unpack):
        inputs, outs, gys = _graph(name)
    for a, b in zip(torch.autograd.grad(outs, inputs, gys, create_graph=True), full):
        _close(a.detach(), b)
    assert all(recorded)


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, *ts):
        return tuple(t.clone() for t in ts)

    @staticmethod
    def backward(ctx, *gs):
        return (None,) * len(gs)


@pytest.mark.parametrize("name", [n for n in OPS if n != "unfold"])    # as torch's own unfold, which passes nothing on
def test_zeros_where_no_gradient_flows_in(name):
    inputs, outs, gys = _graph(name)
    for t, got in zip(inputs, torch.autograd.grad(_NoGradient.apply(*outs), inputs, gys, allow_unused=True)):
        assert got is not None and got.shape == t.shape and not got.any()
    if len(outs) == 1:
        return
    for i in range(len(outs)):          # one of the outputs: the others' gradients count as zeros
        (ia, oa, _), (ib, ob, _) = _graph(name), _graph(name)
        part = torch.autograd.grad(oa[i], ia, gys[i])
        for a, b in zip(part, torch.autograd.grad(ob, ib, [g if j == i else g * 0 for j, g in enumerate(gys)])):
            _close(a, b)
