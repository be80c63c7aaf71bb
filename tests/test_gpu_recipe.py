"""The fused glue of the training recipe (input encoding, loss with correct count, weight-constraint cost and
its gradient) against the same formulas in float64 on the CPU, at the edges of its tiles."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Weights(torch.nn.Module):
    def __init__(self, shapes, gen):
        super().__init__()
        import snntc_amd as snn
        self.layers = torch.nn.ModuleList(
            snn.SNN_dense(r - 1, c, weight=(torch.randn(r, c, generator=gen) / r ** 0.5 + 1.0 / r).numpy()) for r, c in shapes)


@pytest.mark.parametrize("shapes", [[(2, 1)], [(64, 64), (65, 65)], [(63, 10), (785, 64), (130, 129)],
                                    [(3 + i, 5 + i) for i in range(50)]])
def test_constraint_cost_and_gradient(shapes):
    from snntc_amd import train
    model = Weights(shapes, torch.Generator().manual_seed(len(shapes))).to(DEV)
    ws = [l.weight for l in model.layers]
    cost = train.constraint_cost(model, 100.0, 1e-2)
    grads = torch.autograd.grad(cost * 0.5, ws)
    ref = [w.detach().double().cpu().requires_grad_(True) for w in ws]
    want = 100.0 * sum(torch.clamp(1.0 - w.sum(0), min=0.0).mean() for w in ref) + 1e-2 * sum((w * w).mean() for w in ref)
    for g, r in zip(grads, torch.autograd.grad(want * 0.5, ref)):
        assert torch.allclose(g.double().cpu(), r, rtol=1e-5, atol=1e-8)
    assert abs(float(cost) - float(want)) <= 1e-5 * max(1.0, abs(float(want)))


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1025, 70001])
def test_encode_input(n):
    from snntc_amd import train
    x = torch.rand(n + 1, device=DEV)
    for v in (x[:n], x[1:]):                                   # 16-byte aligned, and not
        assert torch.allclose(train.encode_input(v), torch.exp(1.0 - v.double()).float(), rtol=5e-7, atol=0)


@pytest.mark.parametrize("B,J", [(1, 1), (5, 4), (257, 10), (1100, 65), (33, 1000)])
def test_train_step_equals_the_stock_composition(B, J):
    """One step through the fused glue against the same model stepped with stock ops: loss, correct count, weights."""
    import snntc_amd as snn
    from snntc_amd import train
    rng = np.random.default_rng(B + J)
    w = (4.0 / 12 + rng.standard_normal((13, J)) / 12 ** 0.5).astype(np.float32)
    images, labels = torch.rand(B, 12, device=DEV), torch.randint(0, J, (B,), device=DEV)
    fused, stock = (snn.SNN_dense(12, J, weight=w).to(DEV) for _ in range(2))
    loss, correct = train.train_step(fused, torch.optim.SGD(fused.parameters(), lr=0.1), images, labels, J)
    pred = stock(torch.exp(1.0 - images))
    onehot = torch.nn.functional.one_hot(labels, J).float()
    cw = stock.weight
    want = snn.loss_func(logit=pred, label=onehot) + 100.0 * torch.clamp(1.0 - cw.sum(0), min=0.0).mean() + 1e-2 * (cw * cw).mean()
    want.backward()
    assert torch.allclose(loss, want.detach(), rtol=1e-5)
    assert int(correct) == int((torch.argmin(pred, 1) == labels).sum())
    assert torch.allclose(fused.weight, (cw - 0.1 * cw.grad).detach(), rtol=1e-5, atol=1e-6)
    tl, tc = train.test_step(stock, images, labels, J)
    assert torch.allclose(tl, want.detach(), rtol=1e-5) and int(tc) == int(correct)


def test_label_outside_the_classes_is_visible():
    from snntc_amd import _lib
    pred = torch.rand(3, 4, device=DEV)
    w = torch.ones(2, 4, device=DEV)
    loss, _ = _lib.native().recipe_step(pred, torch.tensor([0, 4, 1], device=DEV), [w], 1.0, 1.0, False)
    assert torch.isnan(loss)
