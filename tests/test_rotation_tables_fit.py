"""Circuits with angles per sample hold rotation records and tables per sample; where those would
pass what their 32-bit places can name, the unitaries run as products."""
import pytest

import qandle_amd as qandle
from qandle_amd._engine import fused, jit


def _program(n, layers):
    ops = []
    for _ in range(layers):
        ops += [qandle.RX(q, name=f"x{q}", remapping=None) for q in range(n)]
        ops += [qandle.CNOT(q, (q + 1) % n) for q in range(n)]
    return fused.lower_circuit(qandle.Circuit(ops + [qandle.MeasureProbability()], num_qubits=n).circuit)


@pytest.mark.parametrize("B,rotations", [(2 ** 11, True), (2 ** 21, False)])
def test_tables_that_do_not_fit(B, rotations, monkeypatch):
    monkeypatch.setattr(jit, "kernels_for", lambda sources, names: [])
    n, R, TB = 12, 4, 8
    assert fused.real_rotations(R, TB, B, n)
    prog = _program(n, 8)
    pl = fused.get_plan(prog, R, TB)
    ws = fused.pass_words(prog, pl, B, "cpu")
    kern = fused.specialised_kernels(prog, pl, ws, B, True)
    plan = fused.forward_setup(prog, pl, ws, kern, B, "cpu", None, True)
    assert (kern.schedule is not None) == rotations
    assert plan.nlane <= fused.MAX_TABLE_FLOATS
