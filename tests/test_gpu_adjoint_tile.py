"""Adjoint sweep kernels whose psi and lambda change layout through one tile, against the ones
with a tile each: the same operations on the same values, so the gradients agree bit for bit."""
import pytest
import torch

import qandle_amd as qandle
from qandle_amd import config, workloads
from qandle_amd._engine import fused

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B,R,TB,direct", [(4, 300, 2, 6, False), (9, 5, 4, 8, False), (12, 3, 4, 8, False),
                                             (13, 2, 3, 8, True), (14, 2, 4, 9, False), (15, 2, 4, 8, True)])
def test_one_tile(device, monkeypatch, n, B, R, TB, direct):
    w = workloads.rxryrz_ladder(n=n, B=B, depth=4, seed=n)
    circ = qandle.Circuit(w.layers, num_qubits=n).to(device)
    thetas = [m.theta for m in circ.circuit.layers if getattr(m, "theta", None) is not None]
    wt = torch.randn(B, n, generator=torch.Generator().manual_seed(1)).to(device)
    monkeypatch.setattr(fused, "choose_shape", lambda *a, **k: (R, TB))
    monkeypatch.setattr(config, "SPECIALISE", True)
    out = []
    for opts in ({}, {"one_tile": False}):
        for d in ({}, {"direct_load": True, "direct_store": True}) if direct else ({},):
            monkeypatch.setattr(config, "SPECIALISE_ADJOINT_OPTIONS", {**opts, **d})
            x = w.inputs["x"].to(device).requires_grad_(True)
            out.append(torch.autograd.grad((circ(x=x) * wt).sum(), [x, *thetas]))
    for other in out[1:]:
        assert all(torch.equal(a, b) for a, b in zip(out[0], other))
