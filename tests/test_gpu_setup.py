"""qs_setup (all tables of a call in one launch) against the kernels that make them one by
one (qs_half_angle_coeffs, qs_compose_tables, qs_lane_coeffs, qs_product_factors,
qs_factor_apply), and the probabilities a whole-sample tile's measuring pass writes itself.

Both sides run the same float32 / float64 operations on the same angles; the compiler may
contract the factor products differently, so factors are compared to 4 ulp of 1 and the
tables bit for bit."""
import numpy as np
import pytest
import torch

import qandle_amd as qandle
from oracle import fp64
from qandle_amd._engine import fused
from qandle_amd._engine import lib as L

pytestmark = pytest.mark.gpu


def _circuit(n, names, rot):
    layers = [qandle.AngleEmbedding(name="x", qubits=list(range(0, n, 2)), rotation=rot)]
    for q in range(n):
        layers.append(qandle.RY(q, theta=torch.tensor(0.3 + q), remapping=None))
        if q < names:
            layers.append(qandle.RX(q, name=f"a{q}", remapping=None))
    layers += [qandle.CNOT(q, (q + 1) % n) for q in range(n)]
    layers += [qandle.RZ(q, theta=torch.tensor(1.7 - q), remapping=None) for q in range(n)]
    layers += [qandle.RX(q, name=f"a{q}", remapping=None) for q in range(names)]
    layers += [qandle.CNOT(q + 1, q) for q in range(n - 1)]
    layers += [qandle.RY(0, theta=torch.tensor(0.4), remapping=None), qandle.MeasureProbability()]
    return qandle.Circuit(layers, num_qubits=n)


@pytest.mark.parametrize("n,B,names,rot", [(2, 1, 0, "rx"), (5, 65, 1, "rz"), (6, 3, 6, "ry"), (26, 2, 25, "rx")])
def test_setup_tables(device, n, B, names, rot):
    if names > L.SETUP_MAX_NAMED:  # more names than the launch takes: narrow states, wide inputs only
        n = 26
    circ = _circuit(n, names, rot).to(device)
    prog = fused.lower_circuit(circ.circuit)
    gen = torch.Generator().manual_seed(n)
    kw = {f"a{q}": torch.rand(B, 2, generator=gen).to(device)[:, 0] for q in range(names)}  # strided inputs
    if names:
        kw["a0"] = torch.tensor(0.7, device=device)  # one angle for the whole batch
    kw["x"] = torch.rand((n + 1) // 2, B, generator=gen).to(device).t()
    inp = fused.gather_inputs(prog, circ.circuit, None, kw)
    R, TB = fused.choose_shape(n)
    lead = fused.leading_rotations(prog)
    pl = fused.get_plan(lead[0], R, TB)
    ws = fused.pass_words(lead[0], pl, B, device)
    lanes = sorted({u for _, u, ps in ws.entries if not ps})[::-1]
    tables = fused._leading_tables(prog, lead[1], B, device)
    plan = fused.setup_plan(lead[0], ws, lanes, B, device, tables, True)
    new = lambda c: torch.full((c,), float("nan"), device=device)  # noqa: E731
    cs, utab, ltab, efac = new(2 * plan.total), new(8 * ws.nu), new(16 * len(lanes)), new(4 * B * n)
    a = plan.fill(B, L.ptr(cs), L.ptr(utab), L.ptr(ltab), L.ptr(efac))
    hold = fused.setup_inputs(a, prog, inp)
    L.check(L.load().qs_setup(L.ctypes.byref(a), L.stream_of(cs)), "qs_setup")
    cs0 = fused.build_coeffs(prog, inp)
    utab0, _ = fused.compose_tables(ws, cs0, generators=False)
    ltab0 = new(16 * len(lanes))
    idx = torch.tensor(lanes, dtype=torch.int32, device=device)
    L.check(L.load().qs_lane_coeffs(L.ptr(ltab0), L.ptr(utab0), L.ptr(idx), len(lanes), 0, L.stream_of(cs)), "lanes")
    efac0 = fused.absorb_factors(prog, lead[1], fused.product_factors(prog, inp), cs0, B)
    assert torch.equal(cs, cs0.reshape(-1))
    assert torch.equal(utab, utab0[:8 * ws.nu]) and torch.equal(ltab, ltab0)
    assert (efac - efac0.reshape(-1)).abs().max().item() <= 4 * 2 ** -24
    del hold
    # the adjoint's tables from the half angles
    aw, _ = fused.adjoint_words(prog, fused.get_plan(prog, R, TB), B, device, False)
    ap = fused.setup_plan(prog, aw, None, B, device, dagger=True)
    u1, q1 = new(8 * aw.nu), new(8 * aw.nq)
    a = ap.fill(B, L.ptr(cs0), L.ptr(u1), L.ptr(u1), qtab=L.ptr(q1))
    L.check(L.load().qs_setup(L.ctypes.byref(a), L.stream_of(cs)), "qs_setup")
    u0, q0 = fused.compose_tables(aw, cs0)
    assert torch.equal(u1, u0[:8 * aw.nu]) and torch.equal(q1, q0[:8 * aw.nq])


@pytest.mark.parametrize("n,B", [(2, 1), (3, 257), (5, 65), (8, 1), (8, 33), (11, 3), (12, 5), (13, 2)])
@pytest.mark.parametrize("ring", [True, False])
def test_probabilities_written_by_the_measuring_pass(device, n, B, ring):
    """Widths up to the tile's, batches that leave the last tile part empty; ``ring`` ends the
    circuit in CNOTs (readout parities), else in rotations (the bits themselves)."""
    gen = torch.Generator().manual_seed(100 * n + B)
    x = torch.rand(B, n, generator=gen) * 3
    th = torch.rand(2 * n, generator=gen) * 6
    layers = [qandle.AngleEmbedding(name="x", qubits=list(range(n)), rotation="ry")]
    ops = [("embed", "y", list(range(n)), x.double().numpy())]
    for d in range(2):
        for q in range(n):
            layers.append(qandle.RX(q, theta=th[d * n + q], remapping=None))
            ops.append(("rx", q, float(th[d * n + q])))
        if d == 0 or ring:
            for q in range(n - 1):
                layers.append(qandle.CNOT(q, q + 1))
                ops.append(("cnot", q, q + 1))
    circ = qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n).to(device)
    ref = fp64.measure_prob(fp64.simulate(n, ops), n)
    with torch.no_grad():
        P = circ(x=x.to(device)).cpu().numpy().reshape(B, n)
    assert np.abs(P - ref).max() < 1e-5


@pytest.mark.parametrize("B,sps,pad", [(1, 1, 0), (3, 1, 61), (257, 1, 3), (5, 2, 6), (65, 64, 0), (2, 128, 0), (3, 4096, 64)])
def test_gradient_sums_and_routes(device, B, sps, pad):
    """qs_gradients: shared angles (one row, several rows, none), per-sample inputs with a
    stride, against float64 sums: one rounding to float32 and double sums of at most 2^16 terms."""
    NS = B * sps + pad
    gen = torch.Generator().manual_seed(B + sps)
    part = torch.randn(7, NS, generator=gen)
    groups = [([2], 0, 0), ([], 1, 0), ([6, 0, 3], 2, 0), ([1, 5], 3, 1), ([4], 3 + B, 2), ([], 4 + B, 2)]
    size = 3 + B + 2 * B
    first = np.cumsum([0] + [len(g[0]) for g in groups])
    rows = [r for g in groups for r in g[0]]
    dev = lambda v, t: torch.tensor(v, dtype=t, device=device)  # noqa: E731
    d_first, d_rows = dev(first.tolist(), torch.int32), dev(rows, torch.int32)
    place = dev([v for g in groups for v in g[1:]], torch.int64)
    out = torch.full((size,), float("nan"), device=device)
    gp = part.to(device)
    L.check(L.load().qs_gradients(L.ptr(out), L.ptr(gp), L.ptr(d_first), L.ptr(d_rows), L.ptr(place), len(groups), B, NS,
                                  sps, L.stream_of(out)), "qs_gradients")
    per = part[:, :B * sps].double().reshape(7, B, sps).sum(2) / 2
    ref = torch.zeros(size, dtype=torch.float64)
    for rr, at, stride in groups:
        v = per[rr].sum(0) if rr else torch.zeros(B, dtype=torch.float64)
        if stride:
            ref[at:at + B * stride:stride] = v
        else:
            ref[at] = v.sum()
    err = (out.cpu().double() - ref).abs()
    assert bool((err <= 2.0 ** -23 * ref.abs() + 1e-11).all()), err.max()


@pytest.mark.parametrize("n", [5, 8, 9, 10, 11, 12, 13, 14])
def test_shapes_of_small_and_full_batches_agree(device, n):
    """choose_shape's sides of its lines: a few samples (fewer amplitudes per thread) against the
    oracle, and the same samples inside batches of 2^19 and 2^20 amplitudes and one of a few more
    (other tiles, the last one ragged).  Bars as everywhere: 1e-5 on P, 1e-4 on gradients."""
    gen = torch.Generator().manual_seed(n)
    th = (torch.rand(3 * n, generator=gen) * 6).tolist()
    layers = [qandle.AngleEmbedding(name="x", qubits=list(range(n)))]
    gates = []
    for d in range(3):
        for q in range(n):
            layers.append((qandle.RY, qandle.RX, qandle.RZ)[(q + d) % 3](q, theta=torch.tensor(th[d * n + q]), remapping=None))
            gates.append((("ry", "rx", "rz")[(q + d) % 3], q, float(torch.tensor(th[d * n + q]))))
        for q in range(n):
            layers.append(qandle.CNOT(q, (q + 1 + d) % n))
            gates.append(("cnot", q, (q + 1 + d) % n))
    circ = qandle.Circuit(layers + [qandle.MeasureProbability()], num_qubits=n).to(device)
    few = 3
    x = torch.rand((1 << 20 >> n) + few, n, generator=gen) * 3
    w = torch.randn(x.shape, generator=gen)

    def run(rows):
        with torch.no_grad():
            P = circ(x=x[:rows].to(device))
        xx = x[:rows].to(device).requires_grad_(True)
        (circ(x=xx) * w[:rows].to(device)).sum().backward()
        return P[:few].cpu().numpy(), xx.grad[:few].cpu().numpy()

    ops = [("embed", "x", list(range(n)), x[:few].double().numpy())] + gates
    ref = fp64.measure_prob(fp64.simulate(n, ops), n)
    adj = fp64.adjoint_grads(n, ops, w[:few].double().numpy())[0]
    for rows in (few, 1 << 19 >> n, 1 << 20 >> n, (1 << 20 >> n) + few):
        P, gx = run(rows)
        assert np.abs(P - ref).max() < 1e-5, rows
        assert np.abs(gx - adj).max() < 1e-4, rows
