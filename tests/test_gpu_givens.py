"""Compiled forward passes that apply their unitaries as real rotations between diagonals
(givens), against the float64 oracle and the matrix-core passes: states, probabilities and
kept pass outputs, from |0..0> and from a given state, with shared and per-sample angles.

Tolerance: one unitary changes an amplitude by at most 4 float32 roundings and the errors of
its float32 sine and cosine, below 2^-21 of the norm; the gates' errors add up at most
linearly, and a probability's error is at most twice the state's."""
import math
import random

import numpy as np
import pytest
import torch

import qandle_amd as qandle
from oracle import fp64
from qandle_amd import config
from qandle_amd._engine import fused

pytestmark = pytest.mark.gpu
CORNERS = [0.0, math.pi, -math.pi, math.pi / 2, 2 * math.pi, math.pi / 2 - 1e-4, 3 * math.pi]


def _random(n, B, gates, seed):
    """A circuit, its inputs and the oracle's ops: random rotations (some at the angles where
    a unitary is diagonal or antidiagonal), CNOTs, named per-sample angles."""
    rng = random.Random(seed)
    layers, ops, kw = [], [], {}
    for k in range(gates):
        q = rng.randrange(n)
        if rng.random() < 0.3 and n > 1:
            t = rng.choice([x for x in range(n) if x != q])
            layers.append(qandle.CNOT(q, t))
            ops.append(("cnot", q, t))
            continue
        kind = rng.choice(["rx", "ry", "rz"])
        cls = {"rx": qandle.RX, "ry": qandle.RY, "rz": qandle.RZ}[kind]
        if rng.random() < 0.15:
            x = torch.tensor([rng.uniform(-7, 7) for _ in range(B)])
            kw[f"a{k}"] = x
            layers.append(cls(q, name=f"a{k}", remapping=None))
            ops.append((kind, q, x.double().numpy()))
        else:
            a = torch.tensor(rng.choice(CORNERS) if rng.random() < 0.3 else rng.uniform(-7, 7))
            layers.append(cls(q, theta=a, remapping=None))
            ops.append((kind, q, float(a)))
    return qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n), kw, ops


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("n,B,R,TB", [(3, 5, 3, 8), (6, 70, 4, 8), (9, 3, 4, 9), (12, 2, 4, 8), (13, 3, 4, 9),
                                      (14, 2, 4, 9), (15, 3, 3, 8), (15, 1, 5, 8)])
def test_rotations(device, n, B, R, TB, given):
    gates = 25 * n
    circ, kw, ops = _random(n, B, gates, 7 * n + B)
    circ = circ.to(device)
    prog = fused.lower_circuit(circ.circuit)
    psi0 = None
    if given:
        gen = torch.Generator().manual_seed(n)
        psi0 = torch.view_as_complex(torch.randn(B, 1 << n, 2, generator=gen))
        psi0 = psi0 / psi0.norm(dim=1, keepdim=True)
    inp = fused.gather_inputs(prog, circ.circuit, psi0.to(device) if given else None,
                              {k: v.to(device) for k, v in kw.items()})
    ref = fp64.simulate(n, ops, psi0.numpy().astype(np.complex128) if given else None)
    old, res = (config.SPECIALISE, config.SPECIALISE_OPTIONS), []
    try:
        config.SPECIALISE = True
        for givens in (True, False):
            config.SPECIALISE_OPTIONS = {"givens": givens}
            with torch.no_grad():
                cs = fused.build_coeffs(prog, inp)
                efac = None if given else fused.product_factors(prog, inp)
                marks = {0: None}
                s, p = fused.execute(prog, inp, cs, efac, R, TB, want_state=True)
                s, p = s.clone(), p.clone()
                _s, p1 = fused.execute(prog, inp, cs, efac, R, TB, want_state=False)
                fused._execute(prog, inp, cs, efac, R, TB, want_state=True, marks=marks)
                res.append((s, p, p1.clone(), marks[0]))
    finally:
        config.SPECIALISE, config.SPECIALISE_OPTIONS = old
    tol = gates * 2.0 ** -21
    (s, p, p1, m), (_s0, _p0, _p10, m0) = res
    P = fp64.measure_prob(ref, n)
    err = [np.abs(s.cpu().numpy().reshape(ref.shape) - ref).max(),
           *(np.abs(x.cpu().numpy().reshape(P.shape) - P).max() for x in (p, p1))]
    print(f"n={n} B={B} {R},{TB} given={given}: {err}")
    assert err[0] <= tol and max(err[1:]) <= 2 * tol
    if m0 is not None:
        assert (m - m0).abs().max().item() <= tol


def _phases(n, count, gen):
    """RZ gates on one qubit between CNOTs it controls, on a bit that stays out of the registers
    until RX mixes it: their diagonals all join one flush."""
    ops = [("rx", q, 0.3 + q) for q in range(n)]
    for k in range(count):
        ops += [("rz", 0, float(torch.rand((), generator=gen))), ("cnot", 0, 1 + k % (n - 1)),
                ("rx", 1 + (k + 2) % (n - 1), float(torch.rand((), generator=gen)))]
    return ops + [("rx", q, 0.7 - q) for q in range(n)]


@pytest.mark.parametrize("n,count", [(13, 60), (13, 150), (15, 200)])
def test_many_diagonals(device, n, count):
    cls = {"rx": qandle.RX, "rz": qandle.RZ}
    ops = _phases(n, count, torch.Generator().manual_seed(count))
    layers = [qandle.CNOT(o[1], o[2]) if o[0] == "cnot" else
              cls[o[0]](o[1], theta=torch.tensor(o[2], dtype=torch.float32), remapping=None) for o in ops]
    circ = qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n).to(device)
    prog = fused.lower_circuit(circ.circuit)
    inp = fused.gather_inputs(prog, circ.circuit, None, {})
    old = (config.SPECIALISE, config.SPECIALISE_OPTIONS)
    try:
        config.SPECIALISE, config.SPECIALISE_OPTIONS = True, {"givens": True}
        with torch.no_grad():
            s, _p = fused.execute(prog, inp, fused.build_coeffs(prog, inp), fused.product_factors(prog, inp), 4, 9,
                                  want_state=True)
    finally:
        config.SPECIALISE, config.SPECIALISE_OPTIONS = old
    ref = fp64.simulate(n, ops)
    assert np.abs(s.cpu().numpy().reshape(ref.shape) - ref).max() <= len(ops) * 2.0 ** -21


@pytest.mark.parametrize("n,B,lines", [(12, 2047, False), (12, 2048, True), (14, 511, False), (14, 513, True)])
def test_where_the_rotations_run(n, B, lines):
    R, TB = fused.choose_shape(n, False, B)
    assert fused.real_rotations(R, TB, B, n) == lines
