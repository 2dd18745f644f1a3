"""Programs of one structure share plans, words and tables; their parameters stay their own.
Values that tell circuits apart (angles, remappings, leading rotations, input names) never
come from another circuit's entry."""
import gc

import numpy as np
import pytest
import torch

import qandle_amd as qandle
from oracle import fp64
from qandle_amd import qw_map
from qandle_amd._engine import fused


def _circuit(th, lead="rx", remapping=None, tail="ry", n=4):
    kinds = {"rx": qandle.RX, "ry": qandle.RY}
    layers = [qandle.AngleEmbedding(name="x", qubits=list(range(n)))]
    layers += [kinds[lead](q, theta=th[q], remapping=remapping) for q in range(n)]
    layers += [qandle.CNOT(q, q + 1) for q in range(n - 1)]
    layers += [kinds[tail](q, theta=th[n + q], remapping=remapping) for q in range(n)]
    return qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n)


def _ops(th, x, lead="rx", tail="ry", n=4):
    return ([("embed", "x", list(range(n)), x)] + [(lead, q, float(th[q])) for q in range(n)]
            + [("cnot", q, q + 1) for q in range(n - 1)] + [(tail, q, float(th[n + q])) for q in range(n)])


def _angles(seed, n=4):
    return torch.rand(2 * n, generator=torch.Generator().manual_seed(seed)) * 6


def test_structures_share_and_end_with_their_circuits():
    a, b, c = (_circuit(_angles(s)) for s in (1, 2, 3))
    pa, pb = (fused.lower_circuit(m.circuit) for m in (a, b))
    pc = fused.lower_circuit(_circuit(_angles(3), lead="ry").circuit)
    assert pa.common is pb.common and pc.common is not pa.common
    assert fused.get_plan(pa, 4, 8) is fused.get_plan(pb, 4, 8)
    assert fused.pass_words(pa, fused.get_plan(pa, 4, 8), 2, "cpu") is fused.pass_words(pb, fused.get_plan(pb, 4, 8), 2, "cpu")
    # the programs left after the leading rotations are alike, the leading rotations are not
    ra, rc = fused.leading_rotations(pa)[0], fused.leading_rotations(pc)[0]
    assert [(g.kind, g.pos, g.ctrl) for g in ra.gates] == [(g.kind, g.pos, g.ctrl) for g in rc.gates]
    assert ra.common is not rc.common
    count = len(fused._COMMON)
    del a, b, c, pa, pb, pc, ra, rc
    gc.collect()
    assert len(fused._COMMON) < count


def test_angle_list_follows_the_modules():
    th = _angles(5)
    prog = fused.lower_circuit(_circuit(th).circuit)
    mods = [prog.slots[i].module for i in prog.param_slots]
    assert torch.equal(fused.param_angles(prog, torch.device("cpu")), th) and prog.angles
    with torch.no_grad():
        mods[2].theta.fill_(0.25)
    mods[3].theta = torch.nn.Parameter(torch.tensor([0.5]))          # another shape: the general gather
    got = fused.param_angles(prog, torch.device("cpu"))
    assert got[2] == 0.25 and got[3] == 0.5 and torch.equal(got[4:], th[4:])
    mods[1].remapping = qw_map.tanh                                   # another remapping
    assert torch.allclose(fused.param_angles(prog, torch.device("cpu"))[1], qw_map.tanh(th[1]))
    mods[0].remapping = lambda t: 2 * t                               # any callable
    assert fused.param_angles(prog, torch.device("cpu"))[0] == 2 * th[0]
    long = _circuit(th)
    p2 = fused.lower_circuit(long.circuit)
    fused.param_angles(p2, torch.device("cpu"))
    for i in p2.param_slots:                                          # every shape another one
        p2.slots[i].module.theta = torch.nn.Parameter(p2.slots[i].module.theta.detach().reshape(1))
    out = fused.param_angles(p2, torch.device("cpu"))
    assert torch.equal(out.detach(), th)
    out.sum().backward()
    assert all(p2.slots[i].module.theta.grad.item() == 1 for i in p2.param_slots)


@pytest.mark.gpu
def test_shared_structures_compute_their_own_circuits(device):
    """Same structure with other angles, another leading rotation before the same rest, and a
    circuit built again after its structure's first one is gone; forward and gradients."""
    B, n = 5, 4
    x = torch.rand(B, n, generator=torch.Generator().manual_seed(9)) * 3
    w = torch.randn(B, n, generator=torch.Generator().manual_seed(10))
    first = _circuit(_angles(1)).to(device)
    for seed, lead in ((1, "rx"), (2, "rx"), (3, "ry"), (4, "rx")):
        th = _angles(seed)
        circ = first if seed == 1 else _circuit(th, lead).to(device)
        ops = _ops(th, x.double().numpy(), lead)
        with torch.no_grad():
            P = circ(x=x.to(device))
        assert np.abs(P.cpu().numpy() - fp64.measure_prob(fp64.simulate(n, ops), n)).max() < 1e-5
        circ.zero_grad()
        xx = x.to(device).requires_grad_(True)
        (circ(x=xx) * w.to(device)).sum().backward()
        adj = fp64.adjoint_grads(n, ops, w.double().numpy())
        assert np.abs(xx.grad.cpu().numpy() - adj[0]).max() < 1e-4
        got = [p.grad.item() for p in circ.parameters()]
        ref = [adj[k] for k in range(1, len(ops)) if ops[k][0] != "cnot"]
        assert np.abs(np.array(got) - np.array(ref)).max() < 1e-4
        if seed == 3:
            del circ, first
            gc.collect()
            first = None
