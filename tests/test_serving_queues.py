"""Serving streams and hardware queues: small requests wait behind no large chunk, whichever
streams the process took before."""
import itertools
import time

import pytest
import torch

import qandle_amd as qandle
from qandle_amd import workloads
from qandle_amd._engine import serving


@pytest.mark.parametrize("queues", [1, 2, 3, 4])
@pytest.mark.parametrize("count", [2, 3, 4, 5])
def test_assignment(queues, count):
    """Streams as (queue, number): every way the pool's streams may lie on the queues."""
    behind = lambda a, b: a[0] == b[0]  # noqa: E731
    for lie in itertools.product(range(queues), repeat=5):
        streams = [(q, i) for i, q in enumerate(lie)]
        got = serving.queues_apart((0, "main"), streams, count, behind)
        assert len(got) == count and all(s in streams for s in got)
        used, seen = {s[0] for s in got[1:]}, {0, *lie}
        if len(seen) > 2 or (len(seen) == 2 and 0 in lie):  # main's queue, the small stream's, a large one's
            assert got[0][0] not in used and 0 not in used
            assert len(used) == min(count - 1, len(seen - {0, got[0][0]}))


def _request(rid, n, B, device):
    w = workloads.hardware_efficient(n, B, 4, torch.Generator().manual_seed(rid))
    circ = qandle.Circuit(w.layers, num_qubits=n).to(device)
    return serving.Request(rid, circ, {"x": w.inputs["x"].to(device)})


def _ends_first(launch, busy):
    """Whether what ``launch`` enqueues (it returns its event) ends before a spin on ``busy``."""
    torch.cuda.synchronize()
    end = torch.cuda.Event()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(100 * serving.SPIN)
        end.record(busy)
    ev = launch()
    t0 = time.perf_counter()
    while not ev.query() and not end.query() and time.perf_counter() - t0 < 5:
        pass
    first = ev.query() and not end.query()
    torch.cuda.synchronize()
    return first


@pytest.mark.gpu
@pytest.mark.parametrize("taken", [0, 1, 2, 3])
def test_small_requests_beside_large_chunks(device, taken, monkeypatch):
    monkeypatch.setattr(serving, "_STREAMS", {})
    held = [torch.cuda.Stream(device) for _ in range(taken)]
    eng = serving.ServingEngine(device, cap_bytes=1e9, streams=4, small_work=1e7)
    small = eng.prepare(_request(0, 8, 4, device))
    eng.prepare(_request(1, 16, 64, device))  # a large one: the engine's streams are for both kinds from here
    eng.t0 = time.perf_counter()

    def launch():
        ch = serving._Chunk(small, 0, 4, serving.state_footprint(8, 4, *serving.kernel_shape(8, False)),
                            work=small.work * 4)
        eng._launch(ch)
        return ch.event

    launch().synchronize()
    for s in eng.streams[1:]:
        assert _ends_first(launch, s)
    del held


@pytest.mark.gpu
def test_a_launch_waits_for_the_current_stream_when_it_is_at_work(device):
    eng = serving.ServingEngine(device, cap_bytes=1e9, streams=2)
    req = _request(0, 8, 4, device)
    want = req.circuit(**req.inputs).detach().clone()
    eng.prepare(req)
    x = req.inputs["x"].clone()
    req.inputs["x"].zero_()
    torch.cuda.synchronize()
    torch.cuda._sleep(20 * serving.SPIN)  # the inputs arrive on the current stream while the request is launched
    req.inputs["x"].copy_(x)
    eng.serve([req])
    assert (req.result - want).abs().max().item() < 1e-5
