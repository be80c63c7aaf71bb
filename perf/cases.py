"""The work a user of the SNN-TC ops has them do, as cases that can be timed one by one.

Five kinds, each through the package's public entry points:

  dense   one SNN_dense layer: forward alone, or forward and both gradients (through autograd)
  conv    one SNN_conv layer, likewise; with api "ops" through snncv / snncv_grad on the padded image
  net     a layer stack of snntc_amd.networks, its conv layers chained: inference ("forward"), forward, loss and
          backward ("grad"), or a whole plain-SGD training step ("train")
  recipe  snntc_amd.train.train_step of a small two-conv, two-dense classifier under Adam: input encoding, loss,
          weight-constraint cost, backward, optimizer

A case's sizes are plain numbers; `prepare` makes its inputs from a seed, `run` is one pass.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "snntc-2023_amd"))       # imported from the root of the tree that is measured
import snntc_amd as snn  # noqa: E402
from snntc_amd import networks, train  # noqa: E402

DEVICE = "cuda:0"
MAX_SPIKE_TIME = 1e5
CLASSES = {"mlp": 10, "cifar": 10, "imagenet": 1000}
#: Share of a row's inputs that a neuron takes before it fires, on the inputs and weights drawn below.
CONSUMED = 0.8


def listed():
    return [
        # One request to a served classifier: three dense layers on one image; launches and host work are all there is.
        _net("mlp_forward_b1", "mlp", 1, 784, "forward"),
        # A dense layer in training at an ordinary batch.
        _dense("dense_grad_b128", 128, 784, 800, True, "grad", 0.0),
        # The whole training step of the 784-800-800-10 classifier.
        _net("mlp_train_b256", "mlp", 256, 784, "train"),
        # The example recipe: small strided convs on 28x28 images that are mostly background (heavy ties), Adam.
        {"name": "recipe_train_b128", "kind": "recipe", "batch": 128, "size": 28},
        # Odd sizes, no bias row, and a tenth of the inputs from neurons that never fired.
        _dense("dense_grad_ragged", 333, 1521, 777, False, "grad", 0.1),
        # Bulk inference of a wide dense layer.
        _dense("dense_forward_b4096", 4096, 784, 800, True, "forward", 0.0),
        # One conv layer of an image net, forward and both gradients, through the ops.
        _conv("conv_grad_b64", 64, 32, 32, 64, 64, 3, 1, "SAME", True, "grad", "ops"),
        # A strided VALID conv whose image, channels and filters are multiples of nothing.
        _conv("conv_grad_ragged", 24, 31, 29, 20, 50, 5, 2, "VALID", False, "grad", "layer"),
        # A small batch through the CIFAR-shaped net, as an evaluation or a batching server runs it.
        _net("cifar_forward_b16", "cifar", 16, 32, "forward"),
        # The CIFAR-shaped net's training step.
        _net("cifar_train_b128", "cifar", 128, 32, "train"),
        # One photograph through the ImageNet-shaped net.
        _net("imagenet_forward_b1", "imagenet", 1, 224, "forward"),
        # The ImageNet-shaped net at its training batch: forward, loss, backward.
        _net("imagenet_grad_b32", "imagenet", 32, 224, "grad"),
    ]


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    while True:
        kind = rng.choice(["dense"] * 4 + ["conv"] * 4 + ["net"] * 4 + ["recipe"])
        if kind == "dense":
            c = _dense(None, _log(rng, 1, 4096), _log(rng, 64, 4096), _log(rng, 10, 2048), rng.random() < 0.7,
                       rng.choice(["forward", "grad"]), rng.choice([0.0, 0.0, 0.1]))
        elif kind == "conv":
            k = rng.choice([1, 3, 3, 3, 5, 7])
            c = _conv(None, _log(rng, 1, 64), _log(rng, 7, 112), _log(rng, 7, 112), _channels(rng, 1, 512),
                      _channels(rng, 8, 512), k, 1 if k == 1 else rng.choice([1, 1, 2]), rng.choice(["SAME", "SAME", "VALID"]),
                      rng.random() < 0.7, rng.choice(["forward", "grad", "grad"]), rng.choice(["layer", "ops"]))
        elif kind == "net":
            name = rng.choice(["mlp", "cifar", "imagenet"])
            if name == "mlp":
                c = _net(None, name, _log(rng, 1, 1024), _log(rng, 64, 1024), rng.choice(["forward", "train"]))
            elif name == "cifar":
                c = _net(None, name, _log(rng, 1, 128), rng.randint(24, 40), rng.choice(["forward", "train"]))
            else:
                c = _net(None, name, _log(rng, 1, 32), rng.randint(64, 224), rng.choice(["forward", "grad"]))
        else:
            c = {"kind": "recipe", "batch": _log(rng, 8, 512), "size": rng.randint(16, 40)}
        # within the largest listed step and within what one layer of it holds
        if all(_inputs(l) <= 4608 and l["segments"] * _inputs(l) * l["outputs"] <= 4e9 for l in _layers(c)):
            return c


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    rng = np.random.default_rng(int(seed))
    kind = case["kind"]
    if kind == "dense":
        B, I, J = case["batch"], case["inputs"], case["outputs"]
        layer = snn.SNN_dense(I, J, biasvolt=1.0 if case["bias"] else 0.0,
                              weight=networks.baseline_weight(rng, I, J, case["bias"])).to(DEVICE)
        x = torch.exp(1.0 - _uniform(gen, B, I))
        if case["silent"]:
            x = torch.where(_uniform(gen, B, I) < case["silent"], torch.full_like(x, MAX_SPIKE_TIME), x)
        state = {"layer": layer, "x": x}
        if case["mode"] == "grad":
            x.requires_grad_(True)
            state["upstream"] = _normal(gen, B, J)
    elif kind == "conv":
        B, H, W, C, Kc, k = (case[n] for n in ("batch", "height", "width", "channels", "filters", "kernel"))
        layer = snn.SNN_conv(C, Kc, k, case["stride"], case["padding"], biasvolt=1.0 if case["bias"] else 0.0,
                             weight=networks.baseline_weight(rng, k * k * C, Kc, case["bias"])).to(DEVICE)
        x = torch.exp(_uniform(gen, B, H, W, C))
        state = {"layer": layer, "x": x}
        nh, nw = _out_hw(case)
        if case["api"] == "ops":
            state["x"] = layer.prepare_input(x).contiguous()
            if case["mode"] == "grad":                   # the op takes the gradient of its whole [2B,...] output
                state["upstream"] = torch.cat([_normal(gen, B, nh, nw, Kc), torch.zeros(B, nh, nw, Kc, device=DEVICE)])
        elif case["mode"] == "grad":
            x.requires_grad_(True)
            state["upstream"] = _normal(gen, B, nh, nw, Kc)
    elif kind == "net":
        name, B = case["net"], case["batch"]
        spec = _spec(case)
        shape = (case["size"],) if name == "mlp" else (case["size"], case["size"], 3)
        labels = torch.randint(0, CLASSES[name], (B,), generator=gen, device=DEVICE)
        state = {"net": networks.build(spec, rng=rng, chain=True).to(DEVICE),
                 "x": train.encode_input(_uniform(gen, B, *shape)),
                 "onehot": torch.nn.functional.one_hot(labels, CLASSES[name]).float()}
    else:
        B, size = case["batch"], case["size"]
        model = networks.build(_spec(case), rng=rng).to(DEVICE)
        ink = torch.clamp(_normal(gen, B, size, size, 1) - 0.9, 0.0, 1.0)      # about a fifth of the pixels are not background
        state = {"model": model, "images": ink, "labels": torch.randint(0, 10, (B,), generator=gen, device=DEVICE),
                 # eps as in the optimizer of the framework the recipe comes from
                 "optimizer": torch.optim.Adam(model.parameters(), lr=1e-3, eps=1e-7)}
    state["case"] = dict(case)
    return state


def run(state):
    case = state["case"]
    kind, mode = case["kind"], case.get("mode")
    if kind == "conv" and case["api"] == "ops":
        layer, x = state["layer"], state["x"]
        y = snn.snncv(x, layer.weight.data, layer.Params)
        if mode == "forward":
            return y
        dx, dw, _ = snn.snncv_grad(state["upstream"], x, layer.weight.data, layer.Params, y)
        return y, dx, dw
    if kind in ("dense", "conv"):
        layer, x = state["layer"], state["x"]
        if mode == "forward":
            with torch.no_grad():
                return layer(x)
        y = layer(x)
        dx, dw = torch.autograd.grad(y, (x, layer.weight), state["upstream"])
        return y.detach(), dx, dw
    if kind == "net":
        net, x = state["net"], state["x"]
        if mode == "forward":
            with torch.no_grad():
                return net(x)
        if mode == "grad":
            loss, grads = networks.forward_backward(net, x, state["onehot"])
            return loss, list(grads)
        loss = networks.sgd_train_step(net, x, state["onehot"], 1e-4)
        return loss, [w.detach() for w in net.weights()]
    loss, correct = train.train_step(state["model"], state["optimizer"], state["images"], state["labels"], 10)
    return loss, correct, [w.detach() for w in state["model"].weights()]


def work(case):
    """Bytes: per layer the input, the weights and the outputs once in the forward pass; what the backward pass reads and
    writes once more.  Operations: two multiply-adds per consumed input of a neuron forward, one multiply-add for dX and a
    subtraction and a multiply-add for dW backward."""
    nbytes = flops = 0.0
    backward = case.get("mode") != "forward"
    ops = case.get("api") == "ops"
    for l in _layers(case):
        out, weights = l["segments"] * l["outputs"], (_inputs(l) + l["bias"]) * l["outputs"]
        pairs = CONSUMED * l["segments"] * _inputs(l) * l["outputs"]
        nbytes += 4.0 * (l["in"] + weights + (2 if backward or ops else 1) * out)
        flops += 4.0 * pairs
        if backward:
            nbytes += 4.0 * (3 * out + l["in"] + 2 * weights + (l["in"] if l["dx"] else 0))
            flops += (5.0 if l["dx"] else 3.0) * pairs
    if case["kind"] == "recipe" or case.get("mode") == "train":
        n = sum((_inputs(l) + l["bias"]) * l["outputs"] for l in _layers(case))
        nbytes += 4.0 * n * (7 if case["kind"] == "recipe" else 3)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Everything is 32-bit sums: one layer's results to 1e-5; through a stack of layers a spike time that moves by a
    rounding can change sides of a neighbour's, so the gradients behind it move a little more."""
    return {"rel": 1e-5, "max": 1e-3} if case["kind"] in ("dense", "conv") else {"rel": 1e-4, "max": 1e-2}


# ---- sizes -------------------------------------------------------------------------------------------------------------

def _dense(name, batch, inputs, outputs, bias, mode, silent):
    c = {"kind": "dense", "batch": batch, "inputs": inputs, "outputs": outputs, "bias": bias, "mode": mode, "silent": silent}
    return dict(c, name=name) if name else c


def _conv(name, batch, height, width, channels, filters, kernel, stride, padding, bias, mode, api):
    if padding == "VALID":
        height, width = max(height, kernel), max(width, kernel)
    c = {"kind": "conv", "batch": batch, "height": height, "width": width, "channels": channels, "filters": filters,
         "kernel": kernel, "stride": stride, "padding": padding, "bias": bias, "mode": mode, "api": api}
    return dict(c, name=name) if name else c


def _net(name, net, batch, size, mode):
    c = {"kind": "net", "net": net, "batch": batch, "size": size, "mode": mode}
    return dict(c, name=name) if name else c


def _log(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _channels(rng, low, high):
    """Half of the layers have a channel count made of sixteens, as most nets' do."""
    n = _log(rng, low, high)
    return n if rng.random() < 0.5 or n < 12 else 16 * int(round(n / 16.0))


def _uniform(gen, *shape):
    return torch.rand(shape, generator=gen, device=DEVICE)


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEVICE)


def _out_hw(case):
    if case["padding"] == "SAME":
        return -(-case["height"] // case["stride"]), -(-case["width"] // case["stride"])
    return tuple((case[n] - case["kernel"]) // case["stride"] + 1 for n in ("height", "width"))


def _spec(case):
    """The layer list of a net or recipe case: the package's own, its input layer fitted to the case's size."""
    size = case["size"]
    if case["kind"] == "recipe":
        side = -(-(-(-size // 2)) // 2)
        return [("conv", 1, 8, 3, 2), ("conv", 8, 16, 3, 2), ("flatten",), ("dense", side * side * 16, 64), ("dense", 64, 10)]
    if case["net"] == "mlp":
        return [("dense", size, 800)] + networks.MLP[1:]
    if case["net"] == "cifar":
        side = -(-size // 8)
        return [("dense", side * side * 128, l[2]) if l[0] == "dense" and l[1] == 2048 else l for l in networks.CIFAR]
    return networks.IMAGENET


def _layers(case):
    """The weighted layers of a case: segments, kernel area, input channels, outputs, input tensor size, bias row, wants dX."""
    if case["kind"] == "dense":
        return [{"segments": case["batch"], "area": 1, "c": case["inputs"], "outputs": case["outputs"],
                 "in": case["batch"] * case["inputs"], "bias": int(case["bias"]), "dx": True}]
    if case["kind"] == "conv":
        nh, nw = _out_hw(case)
        return [{"segments": case["batch"] * nh * nw, "area": case["kernel"] ** 2, "c": case["channels"],
                 "outputs": case["filters"], "in": case["batch"] * case["height"] * case["width"] * case["channels"],
                 "bias": int(case["bias"]), "dx": True}]
    out, side, B = [], case["size"], case["batch"]
    for item in _spec(case):
        if item[0] == "conv":
            _, ci, co, k, s = item
            nxt = -(-side // s)
            out.append({"segments": B * nxt * nxt, "area": k * k, "c": ci, "outputs": co, "in": B * side * side * ci,
                        "bias": 1, "dx": bool(out)})
            side = nxt
        elif item[0] == "pool":
            side = -(-side // item[2])
        elif item[0] == "dense":
            out.append({"segments": B, "area": 1, "c": item[1], "outputs": item[2], "in": B * item[1], "bias": 1, "dx": bool(out)})
    return out


def _inputs(layer):
    return layer["area"] * layer["c"]
