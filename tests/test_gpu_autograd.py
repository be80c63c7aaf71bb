"""The differentiable ops as PyTorch sees them.  The native path knows reverse mode over ordinary tensors; with tangents,
transforms, tracers and modes an op has to behave as the torch.autograd.Function it stands for: refuse what has no rule,
record what is traced, and give the same bits."""
import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rand(*shape):
    return torch.exp(torch.rand(*shape, generator=torch.Generator().manual_seed(sum(shape)))).to(DEV)


def _ops():
    """name -> (function of the differentiated inputs, those inputs)"""
    import snntc_amd as snn
    dense = snn.SNN_dense(12, 20).to(DEV)
    same = snn.SNN_conv(3, 8, 3, 1, "SAME").to(DEV)
    valid = snn.SNN_conv(3, 8, 3, 2, "VALID").to(DEV)
    pool = snn.SNN_maxpool2d(2, 2, "SAME")
    label = torch.eye(5, device=DEV)[:4]
    image = _rand(2, 7, 7, 3)

    def weights_of(layer, x):
        return lambda xx, w: torch.func.functional_call(layer, {"weight": w}, (xx,)), (x, layer.weight.detach())

    return {
        "dense": weights_of(dense, _rand(4, 12)),
        "conv_same": weights_of(same, image),
        "conv_valid": weights_of(valid, image),
        "fc": (lambda x, w: snn.SnnFc.apply(x, w, dense.Params), (_rand(4, 12), dense.weight.detach())),
        "cv": (lambda x, w: snn.SnnCv.apply(x, w, valid.Params), (image, valid.weight.detach())),
        "pool": (pool, (image,)),
        "pad": (lambda x: same.prepare_input(x), (image,)),
        "loss": (lambda x: snn.loss_func(logit=x, label=label), (_rand(4, 5),)),
    }


OPS = ["dense", "conv_same", "conv_valid", "fc", "cv", "pool", "pad", "loss"]


@pytest.mark.parametrize("name", OPS)
def test_tangents_and_transforms_are_refused(name):
    f, inputs = _ops()[name]
    for i in range(len(inputs)):
        with fwAD.dual_level():
            args = [fwAD.make_dual(t, torch.ones_like(t)) if i == j else t for j, t in enumerate(inputs)]
            with pytest.raises(NotImplementedError):
                f(*args)
            with torch.no_grad(), pytest.raises(NotImplementedError):
                f(*args)
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: f(*[t if i == j else u for j, u in enumerate(inputs)]).sum())(inputs[i])
    with pytest.raises(RuntimeError):
        torch.func.vmap(f)(*[torch.stack([t, t]) for t in inputs])


class _Watch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("name", OPS)
def test_the_function_and_the_native_node_agree(name):
    f, inputs = _ops()[name]

    def run(watch):
        args = [t.clone().requires_grad_(True) for t in inputs]
        if watch:
            with _Watch():
                out = f(*args)
        else:
            out = f(*args)
        return [out, *torch.autograd.grad(out, args, torch.ones_like(out))], type(out.grad_fn).__name__

    native, node = run(False)
    function, other = run(True)
    assert node != other
    for a, b in zip(native, function):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", ["dense", "conv_valid"])      # (SAME padding computes with sizes a tracer cannot follow)
def test_a_trace_records_the_op(name):
    import snntc_amd as snn
    module = (snn.SNN_dense(12, 20) if name == "dense" else snn.SNN_conv(3, 8, 3, 2, "VALID")).to(DEV)
    x = _rand(4, 12) if name == "dense" else _rand(2, 7, 7, 3)
    with torch.no_grad():
        traced = torch.jit.trace(module, (x,))
        for y in (x, 2.0 - 0.5 * x):
            assert torch.equal(traced(y), module(y))


# ---- the recipe's encoding and weight-constraint cost: stock ops wherever the kernels would lose something ------------

def _stock_cost(weights, k, k2):
    return (k * sum(torch.clamp(1.0 - w.sum(0), min=0.0).mean() for w in weights)
            + k2 * sum(torch.square(w).mean() for w in weights))


class _Held(torch.nn.Module):
    """Something with layers whose weights are whatever tensors it is given."""

    class Layer(torch.nn.Module):
        w_sum_cost = None

        def __init__(self, weight):
            super().__init__()
            self.weight = weight

    def __init__(self, *weights):
        super().__init__()
        self.layers = torch.nn.ModuleList(self.Layer(w) for w in weights)


def _weights():
    return [_rand(13, 20) / 13, _rand(21, 5) / 40]


def test_encoding_keeps_tangents_transforms_and_strides():
    from snntc_amd import train
    x, t = torch.rand(4, 6, device=DEV), torch.rand(4, 6, device=DEV)
    want = torch.exp(1.0 - x)
    with fwAD.dual_level():
        out = fwAD.unpack_dual(train.encode_input(fwAD.make_dual(x, t)))
        assert torch.allclose(out.tangent, -want * t) and torch.allclose(out.primal, want)
    assert torch.allclose(torch.func.vmap(train.encode_input)(x), want)
    assert torch.allclose(torch.func.grad(lambda v: train.encode_input(v).sum())(x), -want)
    assert torch.allclose(torch.jit.trace(train.encode_input, (x,))(t), torch.exp(1.0 - t))
    assert torch.allclose(torch.compile(train.encode_input, backend="eager", fullgraph=True)(x), want)
    assert train.encode_input(x.t()).stride() == x.t().stride() and torch.equal(train.encode_input(x.t()), train.encode_input(x).t())


def test_cost_keeps_tangents_transforms_and_factors():
    from snntc_amd import train
    ws = _weights()

    def cost(*w, k=100.0, k2=1e-2):
        return train.constraint_cost(_Held(*w), k, k2)

    tangents = [torch.rand_like(w) for w in ws]
    grads = torch.func.grad(_stock_cost)(ws, 100.0, 1e-2)
    directional = sum((g * t).sum() for g, t in zip(grads, tangents))
    with fwAD.dual_level():
        out = fwAD.unpack_dual(cost(*[fwAD.make_dual(w, t) for w, t in zip(ws, tangents)]))
        assert torch.allclose(out.tangent, directional, rtol=1e-5)
    for g, want in zip(torch.func.grad(cost, argnums=(0, 1))(*ws), grads):
        assert torch.allclose(g, want, rtol=1e-5)
    many = [torch.stack([w, 2 * w]) for w in ws]
    each = torch.stack([_stock_cost(ws, 100.0, 1e-2), _stock_cost([2 * w for w in ws], 100.0, 1e-2)])
    assert torch.allclose(torch.func.vmap(cost)(*many), each, rtol=1e-5)
    k, k2 = (torch.tensor(v, device=DEV, requires_grad=True) for v in (100.0, 1e-2))
    got = torch.autograd.grad(cost(*ws, k=k, k2=k2), [k, k2])
    for g, want in zip(got, torch.autograd.grad(_stock_cost(ws, k, k2), [k, k2])):
        assert torch.allclose(g, want, rtol=1e-5)


def test_recipe_step_with_a_factor_that_is_a_tensor():
    import snntc_amd as snn
    from snntc_amd import train
    w = torch.rand(13, 4).numpy() / 4
    images, labels = torch.rand(5, 12, device=DEV), torch.randint(0, 4, (5,), device=DEV)
    results = []
    for k in (100.0, torch.tensor(100.0, device=DEV)):
        model = snn.SNN_dense(12, 4, weight=w).to(DEV)
        loss, correct = train.train_step(model, torch.optim.SGD(model.parameters(), lr=0.1), images, labels, 4, weight_k=k)
        results.append((loss, correct, model.weight.detach()))
    for a, b in zip(*results):
        assert torch.allclose(a.float(), b.float(), rtol=1e-5, atol=1e-6)


def test_gradients_of_the_gradient():
    """A penalty on the cost's gradient, and the loss's gradient in its upstream factor: the same second derivatives as the
    stock composition in float64."""
    import snntc_amd as snn
    from snntc_amd import train
    ws = [w.requires_grad_(True) for w in _weights()]
    ref = [w.detach().double().cpu().requires_grad_(True) for w in ws]
    scale, ref_scale = torch.tensor(3.0, device=DEV, requires_grad=True), torch.tensor(3.0, dtype=torch.float64, requires_grad=True)

    def penalty(cost, weights, s):
        first = torch.autograd.grad(cost * s, weights, create_graph=True)
        return [*first, *torch.autograd.grad(sum((g * g).sum() for g in first), [*weights, s])]

    for g, want in zip(penalty(train.constraint_cost(_Held(*ws), 100.0, 1e-2), ws, scale), penalty(_stock_cost(ref, 100.0, 1e-2), ref, ref_scale)):
        assert torch.allclose(g.double().cpu(), want, rtol=1e-5, atol=1e-9)

    times = _rand(4, 5).requires_grad_(True)
    label = torch.eye(5, device=DEV)[:4]
    first, = torch.autograd.grad(snn.loss_func(logit=times, label=label) * scale, [times], create_graph=True)
    by_scale, = torch.autograd.grad((first * first).sum(), [scale])
    assert torch.allclose(by_scale, 2.0 * (first.detach() ** 2).sum() / 3.0, rtol=1e-5)


def test_batched_upstream_gradients_of_cost_and_loss():
    import snntc_amd as snn
    from snntc_amd import train
    ws = [w.requires_grad_(True) for w in _weights()]
    times, label = _rand(4, 5).requires_grad_(True), torch.eye(5, device=DEV)[:4]
    up = torch.tensor([1.0, 0.5, -2.0], device=DEV)
    for out, inputs in ((train.constraint_cost(_Held(*ws)), ws), (snn.loss_func(logit=times, label=label), [times])):
        one = torch.autograd.grad(out, inputs, retain_graph=True)
        for g, want in zip(torch.autograd.grad(out, inputs, up, is_grads_batched=True), one):
            assert torch.allclose(g, up.view(-1, 1, 1) * want, rtol=1e-5)
