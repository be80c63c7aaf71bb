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
