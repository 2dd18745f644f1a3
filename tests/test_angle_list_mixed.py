"""Circuits whose angles are not alike (0-d and one-element parameters, other remappings) take the
general gather at once; a list whose modules changed is made again, or given up."""
import torch

import qandle_amd as qandle
from qandle_amd import qw_map
from qandle_amd._engine import fused

CPU = torch.device("cpu")


def _program(shapes, remaps):
    layers = [qandle.RY(0, theta=torch.full(s, 0.1 + k), remapping=r) for k, (s, r) in enumerate(zip(shapes, remaps))]
    circ = qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=1)
    prog = fused.lower_circuit(circ.circuit)
    return circ, prog, [prog.slots[i].module for i in prog.param_slots]


def test_mixed_angles_take_the_general_gather(monkeypatch):
    tried = []
    gather = fused.AngleList.gather
    monkeypatch.setattr(fused.AngleList, "gather", lambda self, dev: tried.append(1) or gather(self, dev))
    for shapes, remaps in (([(), (1,), ()], [None] * 3), ([(), ()], [None, qw_map.tanh])):
        circ, prog, mods = _program(shapes, remaps)
        for _ in range(2):
            got = fused.param_angles(prog, CPU)
        want = torch.stack([m.remapping(m.theta).reshape(()) for m in mods])
        assert torch.equal(got, want) and prog.angles is False and not tried


def test_a_changed_list_is_made_again_or_given_up():
    circ, prog, mods = _program([()] * 3, [None] * 3)
    fused.param_angles(prog, CPU)
    for m in mods:
        m.theta = torch.nn.Parameter(m.theta.detach().reshape(1))
    assert torch.equal(fused.param_angles(prog, CPU), torch.tensor([0.1, 1.1, 2.1]))
    assert prog.angles and prog.angles.shape == (1,)
    mods[1].theta = torch.nn.Parameter(torch.tensor(0.5))
    assert torch.equal(fused.param_angles(prog, CPU), torch.tensor([0.1, 0.5, 2.1]))
    assert prog.angles is False
