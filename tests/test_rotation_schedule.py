"""The steps of the real-rotation form (givens.Schedule) executed in numpy, against the float64
oracle: tiles of part of a sample and of several, generated and given states, states kept after
some passes, per-sample angles, unitaries that are diagonal or antidiagonal, and runs of
diagonals on bits that stay out of the registers."""
import math
import random

import numpy as np
import pytest
import torch

import qandle_amd as qandle
from oracle import fp64
from qandle_amd._engine import fused, jit
from qandle_amd._engine import givens as GV
from qandle_amd._engine import planner as PL
from tests.fused_emulator import compose
from tests.test_engine_words import coefficients

CORNERS = [0.0, math.pi, -math.pi, math.pi / 2, 2 * math.pi, 3 * math.pi]


def _circuit(n, B, gates, seed, mix):
    rng = random.Random(seed)
    layers, ops, kw = [], [], {}
    for k in range(gates):
        q = rng.randrange(n)
        if rng.random() < 0.35:
            t = rng.choice([x for x in range(n) if x != q])
            layers.append(qandle.CNOT(q, t))
            ops.append(("cnot", q, t))
            continue
        kind = rng.choice(mix)
        cls = {"rx": qandle.RX, "ry": qandle.RY, "rz": qandle.RZ}[kind]
        if rng.random() < 0.2:
            kw[f"a{k}"] = np.array([rng.uniform(-7, 7) for _ in range(B)])
            layers.append(cls(q, name=f"a{k}", remapping=None))
            ops.append((kind, q, kw[f"a{k}"]))
        else:
            a = float(np.float32(rng.choice(CORNERS) if rng.random() < 0.3 else rng.uniform(-7, 7)))
            layers.append(cls(q, theta=torch.tensor(a), remapping=None))
            ops.append((kind, q, a))
    circ = qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n)
    return circ, fused.lower_circuit(circ.circuit), ops, kw


class Split:
    """U = a diag(1, w) R diag(1, g), as the record of a unitary says."""

    def __init__(self, U):
        c, s = abs(U[0, 0]), abs(U[1, 0])
        p, q = (U[0, 0] / c if c else 1), (U[1, 0] / s if s else 1)
        self.g, self.w = np.conj(p * q), q * np.conj(p)
        if s > c:
            self.a, t = s * p, c / s
            self.R = np.array([[t, -1], [1, t]])
        else:
            self.a, t = c * p, s / c
            self.R = np.array([[1, -t], [t, 1]])


def _execute(schedule, passes, n, R, TB, b, psi, utab, cs, generated):
    """Passes over sample b's state (2^n); yields the state after every pass."""
    def unitary(ref, ps):
        return Split(utab[ref + (b if ps else 0)])

    def value(f):
        if f.kind in (GV.ZW, GV.ZNUM):
            c, s = cs[f.ref + (b if f.ps else 0)]
            z = c - 1j * s
            return z if f.kind == GV.ZNUM else np.conj(z) ** 2 / abs(z) ** 2
        u = unitary(f.ref, f.ps)
        return {GV.G: u.g, GV.W: u.w, GV.NUM: u.a}[f.kind]

    records = {k: key for key, k in schedule.records.items()}
    psi = psi.copy()
    if generated and schedule.start:
        psi *= np.prod([value(f) for f, _ in schedule.tables[0]])
    idx = np.arange(1 << n)
    for i, subs in enumerate(passes):
        for sub, (steps, phys, left) in zip(subs, schedule.steps[i]):
            base = idx[np.all([(idx >> p) & 1 == 0 for p in sub.GP], axis=0)]  # the threads
            where = [base + sum(1 << sub.GP[r] for r in range(R) if (j >> r) & 1) for j in range(1 << R)]
            v = [psi[w].copy() for w in where]
            for step in steps:
                if step[0] == "table":
                    for k in range(1 << R):
                        e = 1
                        for f, m in schedule.tables[step[1]]:
                            if f.kind in (GV.NUM, GV.ZNUM) or GV.parity(m & k):
                                e = e * value(f)
                        assert k in step[2] or abs(e - 1) < 1e-12
                        v[k] = v[k] * e
                elif step[0] == "rot":
                    assert records[step[1]][1] == step[2]
                    M = unitary(*records[step[1]]).R
                    for x, y in step[3]:
                        v[x], v[y] = M[0, 0] * v[x] + M[0, 1] * v[y], M[1, 0] * v[x] + M[1, 1] * v[y]
                elif step[0] == "gen":
                    U = utab[step[1] + b]
                    for x, y in step[2]:
                        v[x], v[y] = U[0, 0] * v[x] + U[0, 1] * v[y], U[1, 0] * v[x] + U[1, 1] * v[y]
                elif step[0] == "swap":
                    c = (base >> step[1]) & 1 == 1
                    for x, y in step[2]:
                        v[x], v[y] = np.where(c, v[y], v[x]), np.where(c, v[x], v[y])
                else:
                    z = np.ones(len(base), complex)
                    for f, pos in step[1]:
                        z = np.where((base >> pos) & 1 == 1, z * value(f), z)
                    v = [x * z for x in v]
            for pos, ci, fl in left:
                if not fl & PL.SEG_NOUNAPPLY:
                    c, s = cs[ci + (b if fl & PL.SEG_PER_SAMPLE else 0)]
                    z = np.where((base >> pos) & 1 == 1, c + 1j * s, c - 1j * s)
                    v = [x * z for x in v]
            for j, w in enumerate(where):
                psi[w] = v[phys[j]]
        assert np.abs(psi).max() <= 2.0 ** 34
        yield psi.copy()


@pytest.mark.parametrize("mix", [("rx", "ry", "rz"), ("rz", "rz", "rz", "rx")])
@pytest.mark.parametrize("generated", [True, False])
@pytest.mark.parametrize("n,R,TB", [(3, 3, 6), (5, 4, 6), (7, 2, 3), (8, 3, 3), (8, 4, 2), (9, 4, 3)])
def test_schedule_matches_fp64(n, R, TB, generated, mix):
    B = 2
    for seed in range(4):
        circ, prog, ops, kw = _circuit(n, B, 12 * n + 40 * seed, 100 * n + seed, mix)
        pl = PL.plan(prog.n, prog.gates, R, TB, PL.CostModel(budget=1024.0, min_low=min(2, R + TB - 1)))
        ws = fused.pass_words(prog, pl, B, "cpu")
        words = [w for w, _, _ in ws.host_passes()]
        passes = [PL.decode_pass(w, R, TB) for w in words]
        cs = coefficients(prog, B, kw)
        utab, _ = compose(ws.recipes.numpy(), B, cs, ws.nu, ws.nq)
        last = len(passes) - 1
        psi0 = np.zeros((B, 1 << n), complex)
        psi0[:, 0] = 1
        if not generated:
            g = np.random.default_rng(seed)
            psi0 = g.normal(size=psi0.shape) + 1j * g.normal(size=psi0.shape)
            psi0 /= np.linalg.norm(psi0, axis=1, keepdims=True)
        ref = fp64.simulate(n, ops, psi0)
        kept = random.Random(seed).sample(range(last), min(last, 2))
        for exact in ((), (last,), tuple(sorted({*kept, last}))):
            schedule = jit.rotation_schedule(ws.host_passes(), n, R, TB, generated, exact)
            states = [list(_execute(schedule, passes, n, R, TB, b, psi0[b], utab, cs, generated)) for b in range(B)]
            final = np.stack([s[-1] for s in states])
            assert np.abs(np.abs(final) ** 2 - np.abs(ref) ** 2).max() < 1e-10
            if exact:
                assert np.abs(final - ref).max() < 1e-10
            for i in exact[:-1]:  # a kept state is the one the exact schedule of the passes up to it ends with
                upto = GV.Schedule(passes[:i + 1], R, n < R + TB, generated, (i,))
                for b in range(B):
                    *_, want = _execute(upto, passes[:i + 1], n, R, TB, b, psi0[b], utab, cs, generated)
                    assert np.abs(states[b][i] - want).max() < 1e-10
