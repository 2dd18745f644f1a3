"""Angles and features given as lazily negated views (``z.conj().imag`` shares z's memory, which
holds the numbers with the other sign): the same results as for a materialised copy, bit for bit."""
import ctypes

import pytest
import torch

import qandle_amd as qandle
from qandle_amd._engine import fused
from qandle_amd._engine import lib as L


def _negated(t):
    v = torch.complex(torch.zeros_like(t), -t).conj().imag
    assert v.is_neg() and torch.equal(v, t)
    return v


def _circuit(names, n=3):
    layers = [qandle.AngleEmbedding(name="x", qubits=list(range(n))),
              qandle.RY(0, theta=torch.tensor(0.6), remapping=_negated)]
    layers += [qandle.RX(q % n, name=f"a{q}", remapping=None) for q in range(names)]
    layers += [qandle.CNOT(q, q + 1) for q in range(n - 1)]
    layers += [qandle.RX(q % n, name=f"a{q}", remapping=None) for q in range(names)]
    return qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n)


def _floats(address, count, stride):
    return [ctypes.cast(address + 4 * k * stride, ctypes.POINTER(ctypes.c_float))[0] for k in range(count)]


@pytest.mark.parametrize("names", [2, L.SETUP_MAX_NAMED + 1])
def test_setup_reads_the_negated_numbers(names):
    B, n = 5, 3
    gen = torch.Generator().manual_seed(1)
    named = {f"a{q}": torch.rand(B, generator=gen) for q in range(names)}
    x = torch.rand(B, n, generator=gen)
    circ = _circuit(names)
    prog = fused.lower_circuit(circ.circuit)
    phi = fused.param_angles(prog, torch.device("cpu"))
    inp = fused.Inputs(B, True, torch.device("cpu"), phi, {k: _negated(v) for k, v in named.items()}, _negated(x), None)
    a = L.SetupArgs()
    a.efac = 1  # wanted
    hold = fused.setup_inputs(a, prog, inp)
    flat = _floats(a.phi, a.nphi, 1)
    assert flat[0] == phi[0].item()
    for j, v in enumerate(named.values()):
        got = _floats(a.named[j], B, a.named_stride[j]) if a.nnamed else flat[1 + j * B:1 + (j + 1) * B]
        assert got == v.tolist()
    assert [_floats(a.x + 4 * b * a.x_stride, n, a.x_step) for b in range(B)] == x.tolist()
    del hold


@pytest.mark.gpu
@pytest.mark.parametrize("names", [2, L.SETUP_MAX_NAMED + 1])
def test_circuit(device, names):
    B, n = 5, 3
    gen = torch.Generator().manual_seed(2)
    vals = {f"a{q}": torch.rand(B, generator=gen).to(device) for q in range(names)}
    vals["x"] = torch.rand(B, n, generator=gen).to(device)
    circ = _circuit(names).to(device)
    w = torch.rand(B, n, generator=gen).to(device)
    outs = []
    for make in (lambda t: t, _negated):
        with torch.no_grad():
            P = circ(**{k: make(v) for k, v in vals.items()})
        ins = {k: v.clone().requires_grad_(True) for k, v in vals.items()}
        out = circ(**{k: make(v) for k, v in ins.items()})
        outs.append([P, out.detach(), *torch.autograd.grad((out * w).sum(), list(ins.values()))])
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.gpu
def test_operators_alone(device):
    B, n = 4, 3
    gen = torch.Generator().manual_seed(3)
    st = torch.randn(B, 2 ** n, dtype=torch.complex64, generator=gen).to(device)
    phi = torch.rand(B, generator=gen).to(device)
    for op in (qandle.RX(1, name="a", remapping=None), qandle.Controlled(0, qandle.RY(2, name="a", remapping=None))):
        m = op.build(num_qubits=n).to(device)
        for v in (phi, phi[0]):
            assert torch.equal(m(st, a=v), m(st, a=_negated(v)))
