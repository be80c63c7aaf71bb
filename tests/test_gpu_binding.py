"""Properties of the native autograd nodes that their numbers do not show: what a saved output does after an in-place change,
graphs walked twice, saved-tensor hooks, inputs with other strides, backward passes on another stream, several threads."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rand(*shape, seed=0):
    return torch.exp(torch.rand(*shape, generator=torch.Generator().manual_seed(seed + sum(shape)))).to(DEV)


def _layers():
    """name -> (layer, input shape)"""
    import snntc_amd as snn
    return {"dense": (snn.SNN_dense(30, 40).to(DEV), (6, 30)),
            "head": (snn.SNN_dense(30, 10).to(DEV), (6, 30)),
            "conv_same": (snn.SNN_conv(8, 16, 3, 1, "SAME").to(DEV), (2, 9, 9, 8)),
            "conv_valid": (snn.SNN_conv(5, 16, 3, 2, "VALID").to(DEV), (2, 9, 9, 5)),
            "pool": (snn.SNN_maxpool2d(2, 2, "SAME"), (2, 9, 9, 8))}


LAYERS = ["dense", "head", "conv_same", "conv_valid", "pool"]


def _inputs(layer, x):
    return [x, *layer.parameters()]


def _grads(layer, x, y):
    return torch.autograd.grad(y, _inputs(layer, x), torch.cos(torch.arange(y.numel(), device=DEV).float()).view_as(y))


@pytest.mark.parametrize("name", ["dense", "head", "conv_same", "conv_valid"])
def test_an_output_changed_in_place_is_noticed(name):
    """The spike times handed out are the first half of the output the node has saved."""
    layer, shape = _layers()[name]
    y = layer(_rand(*shape).requires_grad_(True))
    with torch.no_grad():
        y.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


@pytest.mark.parametrize("name", LAYERS)
def test_a_graph_is_walked_twice_or_freed(name):
    layer, shape = _layers()[name]
    x = _rand(*shape).requires_grad_(True)
    y = layer(x)
    up = torch.ones_like(y)
    first = torch.autograd.grad(y, _inputs(layer, x), up, retain_graph=True)
    second = torch.autograd.grad(y, _inputs(layer, x), up)
    assert all(torch.equal(a, b) for a, b in zip(first, second))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, _inputs(layer, x), up)


@pytest.mark.parametrize("name", LAYERS)
def test_saved_tensor_hooks_see_what_is_saved(name):
    layer, shape = _layers()[name]
    x = _rand(*shape).requires_grad_(True)
    want = _grads(layer, x, layer(x))
    packed = []

    def pack(t):
        packed.append(tuple(t.shape))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        y = layer(x)
    assert len(packed) == (1 if name == "pool" else 3)
    assert all(torch.equal(a, b) for a, b in zip(_grads(layer, x, y), want))


@pytest.mark.parametrize("name", LAYERS)
def test_inputs_with_other_strides(name):
    layer, shape = _layers()[name]
    x = _rand(*shape)
    plain = x.clone().requires_grad_(True)
    y = layer(plain)
    want = _grads(layer, plain, y)
    order = list(range(len(shape)))[::-1]
    leaf = x.permute(order).contiguous().requires_grad_(True)
    turned = leaf.permute(order)                            # (reversing twice is the identity)
    assert not turned.is_contiguous()
    z = layer(turned)
    assert torch.equal(z, y)
    got = _grads(layer, leaf, z)
    assert torch.equal(got[0].permute(order), want[0]) and all(torch.equal(a, b) for a, b in zip(got[1:], want[1:]))


@pytest.mark.parametrize("name", LAYERS)
def test_forward_and_backward_on_different_streams(name):
    layer, shape = _layers()[name]
    x = _rand(*shape).requires_grad_(True)
    want = _grads(layer, x, layer(x))
    side = torch.cuda.Stream()
    for _ in range(5):
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y = layer(x)
        torch.cuda.current_stream().wait_stream(side)
        got = _grads(layer, x, y)
        del y
        junk = [torch.full((4096,), -1.0, device=DEV) for _ in range(8)]     # memory given back is taken and overwritten
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        del junk


def test_threads_with_streams_of_their_own():
    """Four threads, each on its own stream, run layers forward and backward with the interpreter lock released."""
    layers = _layers()
    work = [(name, seed) for seed in range(2) for name in LAYERS]
    want = {}
    for name, seed in work:
        layer, shape = layers[name]
        x = _rand(*shape, seed=seed).requires_grad_(True)
        y = layer(x)
        want[name, seed] = [y.detach(), *_grads(layer, x, y)]
    torch.cuda.synchronize()
    failures = []

    def run(turn):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for k in range(20):
                    name, seed = work[(k + turn * 3) % len(work)]
                    layer, shape = layers[name]
                    x = _rand(*shape, seed=seed).requires_grad_(True)
                    y = layer(x)
                    got = [y.detach(), *_grads(layer, x, y)]
                    stream.synchronize()
                    if not all(torch.equal(a, b) for a, b in zip(got, want[name, seed])):
                        failures.append((turn, k, name, seed))
        except Exception as e:                              # noqa: BLE001 -- reported by the main thread
            failures.append((turn, repr(e)))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failures


def test_inference_mode_and_no_grad():
    for name in LAYERS:
        layer, shape = _layers()[name]
        x = _rand(*shape)
        y = layer(x)
        with torch.inference_mode():
            assert torch.equal(layer(x), y)
        with torch.no_grad():
            z = layer(x.requires_grad_(True))
            assert torch.equal(z, y) and not z.requires_grad
