"""Serving runs one form of the pass kernels for every batch: results do not depend on how a
request is split, and what was compiled ahead is what runs."""
import pytest
import torch

import qandle_amd as qandle
from qandle_amd import workloads
from qandle_amd._engine import fused, jit, serving


def _request(n, B, device):
    w = workloads.hardware_efficient(n, B, 4, torch.Generator().manual_seed(n))
    return serving.Request(0, qandle.Circuit(w.layers, num_qubits=n).to(device), {"x": w.inputs["x"].to(device)})


@pytest.mark.parametrize("n,B", [(4, 2 ** 19), (12, 2048), (13, 1024)])
def test_prepared_kernels_are_the_compiled_ones(n, B, monkeypatch):
    monkeypatch.setattr(jit, "kernels_for", lambda sources, names: [])
    code = []
    monkeypatch.setattr(jit, "_code_for", lambda src: code.append(src) or b"")
    req = _request(n, B, "cpu")
    prog = fused.lower_circuit(req.circuit.circuit)
    serving._compile_worker([serving._spec(prog)])
    R, TB = serving.kernel_shape(n, True)
    built = []
    monkeypatch.setattr(fused, "forward_setup", lambda prog, pl, ws, kern, *a, **k: built.append(kern))
    eng = serving.ServingEngine.__new__(serving.ServingEngine)
    eng.device, eng.cap, eng.max_chunk_frac, eng.small_work = torch.device("cpu"), 10 ** 12, 1.0, float("inf")
    eng.compiled_from, eng.warm = 2, True
    eng.prepare(req)
    assert req.compiled and len(built) == 1
    assert "\n\n".join(built[0].sources) == code[0]


@pytest.mark.gpu
@pytest.mark.parametrize("n,B", [(4, 2 ** 19 + 5), (12, 2049)])
def test_split_requests_give_the_same_bits(device, n, B):
    got = []
    for cap in (1e9, serving.state_footprint(n, B // 3, *serving.kernel_shape(n, True)) * 4.0):
        eng = serving.ServingEngine(device, cap_bytes=cap, streams=2, compiled_from_qubits=4)
        req = eng.prepare(_request(n, B, device))
        got.append((len(req.chunks), eng.serve([req])[0].result))
    assert got[0][0] == 1 and got[1][0] > 1
    assert torch.equal(got[0][1], got[1][1])
