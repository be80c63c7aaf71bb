"""The training-step glue of the reference's example scripts, for models built from the SNN layers:
input encoding, the weight-constraint cost, one Adam/SGD step and the evaluation step
(snntc-mnist.py:55-59, 73-96).  On a ROCm device the encoding, the loss with its count of correct samples
and the weight-constraint cost with its gradient are five kernels (csrc/recipe.hip).  Everything else, and
all of it on other devices and types, with tangents, transforms or tracers at work, or with tensors as cost
factors, is stock PyTorch around the gfx950 ops.  Weights are saved and restored with ``model.state_dict()``
/ ``load_state_dict`` (the reference uses Keras ``save_weights``, snntc-cifar10.py:255-259).
"""
import torch

from ._lib import native
from .layers import loss_func


def encode_input(images):
    """Pixel intensities in [0,1] -> spike times z = exp(1 - x) >= 1 (snntc-mnist.py:75)."""
    if (images.is_cuda and images.dtype == torch.float32 and not (images.requires_grad and torch.is_grad_enabled())
            and not torch.compiler.is_compiling() and native().plain(images) and images.is_contiguous()):
        return native().encode_time(images)
    return torch.exp(1.0 - images)


def snn_layers(model):
    return [m for m in model.modules() if hasattr(m, "w_sum_cost") and hasattr(m, "weight")]


def _fused_weights(layers, weight_k, weight_k2, device=None):
    """The layers' weights as a list if the fused cost kernels take them (contiguous float32 matrices on one
    ROCm device, no tensor twice, nothing but reverse mode to carry derivatives; constant factors), else None."""
    weights = [l.weight for l in layers]
    if isinstance(weight_k, torch.Tensor) or isinstance(weight_k2, torch.Tensor) or torch.compiler.is_compiling():
        return None
    for w in weights:
        if not (isinstance(w, torch.Tensor) and w.is_cuda and w.dtype == torch.float32 and w.dim() == 2 and native().plain(w)
                and w.is_contiguous() and w.device == (device or weights[0].device) and w.numel()):
            return None
    return weights if weights and len({w.data_ptr() for w in weights}) == len(weights) else None


def constraint_cost(model, weight_k=100.0, weight_k2=1e-2):
    """K * sum_l mean(max(0, 1 - sum_i w_ij)) + K2 * sum_l mean(w^2)  (snntc-mnist.py:55-59)."""
    layers = snn_layers(model)
    weights = _fused_weights(layers, weight_k, weight_k2)
    if weights is not None:
        return native().constraint_cost(weights, weight_k, weight_k2)
    wsc = sum(torch.mean(torch.clamp(1.0 - torch.sum(l.weight, 0), min=0.0)) for l in layers)
    l2 = sum(torch.mean(torch.square(l.weight)) for l in layers)
    return weight_k * wsc + weight_k2 * l2


def predictions_to_classes(predictions):
    """The earliest output spike is the predicted class (snntc-mnist.py:83)."""
    return torch.argmin(predictions, dim=1)


def _recipe_weights(model, predictions, labels, num_classes, weight_k, weight_k2):
    """The weights for the fused loss and cost of a step, or None where the step has to go through stock ops:
    other devices and types, tied weights, hooks that want to see a weight's whole gradient."""
    if not (predictions.is_cuda and predictions.dtype == torch.float32 and predictions.dim() == 2
            and predictions.shape[1] == num_classes and predictions.numel() and labels.dtype == torch.int64
            and labels.device == predictions.device and labels.shape == predictions.shape[:1]
            and native().plain(predictions, labels)):
        return None
    weights = _fused_weights(snn_layers(model), weight_k, weight_k2, predictions.device)
    if weights is None or any(w._backward_hooks or w._post_accumulate_grad_hooks or not w.is_leaf for w in weights):
        return None
    return weights


def train_step(model, optimizer, images, labels, num_classes, weight_k=100.0, weight_k2=1e-2):
    """One optimisation step on a batch of images in [0,1]; returns (loss, number of correct samples)."""
    inputs = encode_input(images)
    optimizer.zero_grad(set_to_none=True)
    predictions = model(inputs)
    weights = _recipe_weights(model, predictions, labels, num_classes, weight_k, weight_k2)
    if weights is not None and predictions.requires_grad:
        loss, correct = native().recipe_step(predictions, labels, weights, weight_k, weight_k2, True)
        optimizer.step()
        return loss, correct
    onehot = torch.nn.functional.one_hot(labels, num_classes).to(inputs.dtype)
    loss = loss_func(logit=predictions, label=onehot) + constraint_cost(model, weight_k, weight_k2)
    loss.backward()
    optimizer.step()
    correct = (predictions_to_classes(predictions.detach()) == labels).sum()
    return loss.detach(), correct


@torch.no_grad()
def test_step(model, images, labels, num_classes, weight_k=100.0, weight_k2=1e-2):
    inputs = encode_input(images)
    predictions = model(inputs)
    weights = _recipe_weights(model, predictions, labels, num_classes, weight_k, weight_k2)
    if weights is not None:
        return native().recipe_step(predictions, labels, weights, weight_k, weight_k2, False)
    onehot = torch.nn.functional.one_hot(labels, num_classes).to(inputs.dtype)
    loss = loss_func(logit=predictions, label=onehot) + constraint_cost(model, weight_k, weight_k2)
    return loss, (predictions_to_classes(predictions) == labels).sum()
