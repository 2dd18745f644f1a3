"""A tile shape that the library does not take is refused on the host, before anything is
launched into a workspace that no size query could size."""
import pytest
import torch

import qandle_amd as qandle
from qandle_amd._engine import backward, fused
from qandle_amd._engine.lib import EngineError


def _program(n):
    layers = [qandle.AngleEmbedding(name="x", qubits=list(range(n)))]
    layers += [qandle.RY(q, theta=torch.tensor(0.3), remapping=None) for q in range(n)]
    layers += [qandle.CNOT(q, (q + 1) % n) for q in range(n)] + [qandle.MeasureProbability()]
    return fused.lower_circuit(qandle.Circuit(layers, num_qubits=n).circuit)


@pytest.mark.parametrize("R,TB", [(3, 5), (6, 6), (5, 11), (0, 8)])
def test_refused(R, TB):
    n, B, cpu = 14, 4, torch.device("cpu")
    prog = _program(n)
    with pytest.raises(EngineError, match="unsupported shape"):
        backward._adjoint_call(prog, R, TB, fused.GRAD_COST, B, cpu, True, False, True, True)
    with pytest.raises(EngineError, match="unsupported shape"):
        fused._forward_call(prog, R, TB, fused.DEFAULT_COST, B, cpu, True, False, False, True, None, True, (), None)
