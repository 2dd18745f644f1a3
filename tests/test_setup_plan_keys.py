"""A setup plan fills the tables of one set of kernels: a program whose first pass generates its
state in one call and reads a given one in the next gets a plan for each."""
import pytest
import torch

import qandle_amd as qandle
from qandle_amd import config
from qandle_amd._engine import fused, jit


def _program(n):
    """No leading rotations: every qubit is in a CNOT first."""
    layers = [qandle.CNOT(q, q + 1) for q in range(n - 1)]
    for d in range(3):
        for q in range(n):
            layers += [qandle.RX(q, theta=torch.tensor(0.3 + q), remapping=None),
                       qandle.RZ(q, theta=torch.tensor(0.7 - q), remapping=None)]
        layers += [qandle.CNOT(q, (q + 1) % n) for q in range(n)]
    return qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n)


def _kernels(prog, pl, ws, B, generated, monkeypatch):
    """The kernels' tables without their code objects (nothing is compiled or loaded)."""
    monkeypatch.setattr(jit, "kernels_for", lambda sources, names: [])
    return fused.specialised_kernels(prog, pl, ws, B, generated)


def _words(plan):
    return plan.keep[1].tolist()


def test_generated_and_given_first_pass(monkeypatch):
    n, B, R, TB = 13, 1024, 4, 9
    circ = _program(n)
    prog = fused.lower_circuit(circ.circuit)
    pl = fused.get_plan(prog, R, TB)
    ws = fused.pass_words(prog, pl, B, "cpu")
    plans, fresh = [], []
    for generated in (True, False):
        kern = _kernels(prog, pl, ws, B, generated, monkeypatch)
        assert kern.schedule is not None
        plans.append(fused.forward_setup(prog, pl, ws, kern, B, "cpu", None, False))
        fresh.append(fused.setup_plan(prog, ws, None, B, "cpu", kern=kern))
    assert _words(fresh[0]) != _words(fresh[1])
    for got, want in zip(plans, fresh):
        assert _words(got) == _words(want) and got.nlane == want.nlane


@pytest.mark.gpu
def test_one_program_generated_then_given(device, monkeypatch):
    """Tables made by the caller, as the autotuner times them: from |0..0> and then from a state."""
    n, B, R, TB = 13, 1024, 4, 9
    circ = _program(n).to(device)
    prog = fused.lower_circuit(circ.circuit)
    monkeypatch.setattr(config, "SPECIALISE", True)
    psi0 = torch.zeros(B, 1 << n, dtype=torch.complex64, device=device)
    psi0[:, 0] = 1
    with torch.no_grad():
        inp = fused.gather_inputs(prog, circ.circuit, psi0, {})
        cs, efac = fused.build_coeffs(prog, inp), fused.product_factors(prog, inp)
        zero = fused.Inputs(B, True, inp.device, inp.phi_param, inp.named, None, None)
        _s, want = fused.execute(prog, zero, cs, efac, R, TB, want_state=False)
        _s, got = fused.execute(prog, inp, cs, None, R, TB, want_state=False)
    # equal up to the order of the same float32 roundings: 2^-21 of the norm per gate, twice in a probability
    assert (got - want).abs().max().item() <= 2 * len(prog.gates) * 2.0 ** -21
