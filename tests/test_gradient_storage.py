"""The gradients of one backward pass are tensors of their own: one that autograd saved stays
valid when another is changed in place (a cleared or clipped gradient)."""
import pytest
import torch

import qandle_amd as qandle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("change", ["theta", "named", "features"])
def test_changing_one_gradient_leaves_the_others_versions(device, change):
    B, n = 6, 4
    layers = [qandle.AngleEmbedding(name="x", qubits=list(range(n)))]
    layers += [qandle.RY(q, theta=torch.tensor(0.3 + q), remapping=None) for q in range(n)]
    layers += [qandle.CNOT(q, q + 1) for q in range(n - 1)] + [qandle.RX(0, name="a", remapping=None)]
    circ = qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n).to(device)
    theta = [p for k, p in circ.named_parameters() if not circ.get_submodule(k.rsplit(".", 1)[0]).named]
    leaves = {"features": torch.rand(B, n, device=device).requires_grad_(True),
              "named": torch.rand(B, device=device).requires_grad_(True)}
    circ(x=leaves["features"], a=leaves["named"]).square().sum().backward()
    grads = {"theta": theta[0].grad, **{k: v.grad for k, v in leaves.items()}}
    kept = {k: g.clone() for k, g in grads.items()}
    scale = torch.ones((), device=device, requires_grad=True)
    later = sum((g * scale).sum() for k, g in grads.items() if k != change)  # saves the other gradients
    grads[change].zero_()
    later.backward()
    assert torch.allclose(scale.grad, sum(g.sum() for k, g in kept.items() if k != change))
    assert all(torch.equal(grads[k], kept[k]) for k in grads if k != change)
