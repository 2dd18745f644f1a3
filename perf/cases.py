"""Performance cases of the engine: the calls a user of the package makes, over the range of sizes they are made at.

Kinds of case:

* ``forward``   inference of an embedding circuit without gradients (``Circuit.__call__``): features in, P(qubit = 0) out
* ``train``     one training step's forward + backward of the same circuits: gradients of the inputs and every angle
* ``reupload``  a training step of a data re-uploading circuit (named per-sample rotation inputs)
* ``amplitude`` AmplitudeEmbedding -> StronglyEntanglingLayer -> MeasureJointProbability, forward + backward
* ``qconv``     forward + backward of a QConv layer over a batch of images
* ``gates``     a circuit of operators outside the fused program (Controlled, U, Reset), run operator by operator
* ``uneven``    forward + backward of a batch of different circuits (``UnevenBatch``, one captured graph)
* ``serve``     a burst of requests through the serving engine, until the last result is there

Circuit families (``qandle_amd.workloads``): ``ring`` (RY + CNOT ring), ``ladder`` (RX, RY, RZ + CNOT ladder) and
``hea`` (RY, RZ + CNOT ring, the serving requests' ansatz).
"""
import math

import numpy as np
import torch

import qandle_amd as qandle
from qandle_amd import workloads
from qandle_amd._engine import serving
from qandle_amd._engine.uneven import UnevenBatch

DEV = "cuda:0"


def listed():
    return [
        # a small classifier's inference call: bound by launches and host time
        {"name": "fwd_ring_n8_b32", "kind": "forward", "family": "ring", "n": 8, "B": 32, "depth": 4},
        # the package's headline benchmark workload
        {"name": "fwd_ladder_n20_b64", "kind": "forward", "family": "ladder", "n": 20, "B": 64, "depth": 10},
        # a wide register with few samples
        {"name": "fwd_ladder_n24_b4", "kind": "forward", "family": "ladder", "n": 24, "B": 4, "depth": 10},
        # an ordinary width with an odd batch
        {"name": "fwd_hea_n17_b11", "kind": "forward", "family": "hea", "n": 17, "B": 11, "depth": 7},
        # a training step of the small classifier
        {"name": "train_ring_n8_b32", "kind": "train", "family": "ring", "n": 8, "B": 32, "depth": 4},
        # the package's gradient benchmark workload
        {"name": "train_ladder_n16_b256", "kind": "train", "family": "ladder", "n": 16, "B": 256, "depth": 20},
        # data re-uploading: every sample has its own rotations
        {"name": "train_reupload_n11_b75", "kind": "reupload", "n": 11, "B": 75, "depth": 5},
        # amplitude-encoded features, the whole distribution read out
        {"name": "train_amplitude_n13_b100", "kind": "amplitude", "n": 13, "B": 100, "depth": 4, "features": 6000},
        # a quantum convolution layer on small images
        {"name": "train_qconv_b8_c3_32x32", "kind": "qconv", "b": 8, "c_in": 3, "c_out": 8, "k": 3, "h": 32, "w": 32,
         "depth": 2},
        # operators outside the fused program, one kernel each way per operator
        {"name": "train_gates_n18_b8", "kind": "gates", "n": 18, "B": 8, "depth": 4},
        # many small different circuits (a search over ansaetze)
        {"name": "train_uneven_256", "kind": "uneven", "count": 256, "mix": 3, "n_hi": 18},
        # a burst of requests at a server
        {"name": "serve_24", "kind": "serve", "count": 24, "mix": 4, "n_hi": 20, "b_max": 24},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    cap = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["forward", "forward", "forward", "train", "train", "reupload", "amplitude", "qconv", "gates",
                           "uneven", "serve"])
        if kind in ("forward", "train"):
            n = rng.randint(2, 24 if kind == "forward" else 20)
            top = 2 ** 26 if kind == "forward" else 2 ** 24
            c = {"kind": kind, "family": rng.choice(["ring", "ladder", "hea"]), "n": n,
                 "B": _log_int(rng, 1, min(4096, max(1, top >> n))), "depth": rng.randint(1, 12)}
        elif kind == "reupload":
            n = rng.randint(2, 14)
            c = {"kind": kind, "n": n, "B": _log_int(rng, 2, min(2000, max(2, 2 ** 20 >> n))), "depth": rng.randint(1, 8)}
        elif kind == "amplitude":
            n = rng.randint(2, 16)
            c = {"kind": kind, "n": n, "B": _log_int(rng, 1, min(2048, max(1, 2 ** 21 >> n))), "depth": rng.randint(1, 5),
                 "features": rng.randint(max(1, 2 ** n // 2), 2 ** n)}
        elif kind == "qconv":
            c = {"kind": kind, "b": rng.randint(1, 16), "c_in": rng.randint(1, 4), "c_out": rng.randint(2, 16),
                 "k": rng.choice([2, 3]), "h": rng.randint(5, 32), "w": rng.randint(5, 32), "depth": rng.randint(1, 3)}
        elif kind == "gates":
            n = rng.randint(4, 20)
            c = {"kind": kind, "n": n, "B": _log_int(rng, 1, min(256, max(1, 2 ** 22 >> n))), "depth": rng.randint(1, 5)}
        elif kind == "uneven":
            c = {"kind": kind, "count": _log_int(rng, 8, 256), "mix": rng.randint(10, 10 ** 6), "n_hi": rng.randint(8, 18)}
        else:
            c = {"kind": kind, "count": rng.randint(4, 24), "mix": rng.randint(10, 10 ** 6), "n_hi": rng.randint(12, 20),
                 "b_max": rng.randint(2, 24)}
        if _cost(c) <= cap:
            return c


# ---------------------------------------------------------------------------------------------------------------------
# circuits, as gate lists: ("rx" | "ry" | "rz", qubit, angle index), ("named", kind, qubit, name), ("cnot", control, target)
# ---------------------------------------------------------------------------------------------------------------------
FAMILIES = {"ring": (("ry",), True), "ladder": (("rx", "ry", "rz"), False), "hea": (("ry", "rz"), True)}


def _family(family, n, depth):
    kinds, ring = FAMILIES[family]
    ops, k = [], 0
    for _ in range(depth):
        for q in range(n):
            for kd in kinds:
                ops.append((kd, q, k))
                k += 1
        for q in range(n if ring and n > 1 else n - 1):
            ops.append(("cnot", q, (q + 1) % n))
    return ops, k


def _reupload(n, depth):
    ops, k = [], 0
    for _ in range(depth):
        ops += [("named", "rx", q, f"x{q}") for q in range(n)]
        for kd in ("ry", "rz"):
            for q in range(n):
                ops.append((kd, q, k))
                k += 1
        ops += [("cnot", q, (q + 1) % n) for q in range(n if n > 1 else 0)]
    return ops, k


def _sel(n, depth):
    ops, k = [], 0
    for d in range(depth):
        for q in range(n):
            for kd in ("rz", "ry", "rz"):
                ops.append((kd, q, k))
                k += 1
        off = d % (n - 1) if n > 1 else 0
        ops += [("cnot", q, (q + 1 + off) % n) for q in range(n if n > 1 else 0)]
    return ops, k


def _gates(n, depth):
    """Operators outside the fused program: a custom gate, controlled rotations, CZ, SWAP and a final Reset."""
    ops, k = [], 0
    for d in range(depth):
        for q in range(n):
            ops.append(("ry" if (q + d) % 2 else "rx", q, k))
            k += 1
        ops.append(("u", (3 * d + 1) % n))
        for q in range(0, n - 1, 3):
            ops.append(("ctrl", q, "ry" if q % 2 else "rz", q + 1, k))
            k += 1
        ops += [("cz", 0, n - 1), ("swap", 1, n - 2)] if n > 3 else [("cz", 0, n - 1)]
        ops += [("cnot", q, q + 1) for q in range(d % 2, n - 1, 2)]
    ops.append(("reset", n // 2))
    return ops, k


U_MATRIX = np.linalg.qr(np.array([[0.6 + 0.2j, -0.3 + 0.5j], [0.1 - 0.7j, 0.4 + 0.3j]]))[0].astype(np.complex64)
CLASS = {"rx": qandle.RX, "ry": qandle.RY, "rz": qandle.RZ}


def _layers(ops, theta):
    out = []
    for op in ops:
        if op[0] == "cnot":
            out.append(qandle.CNOT(op[1], op[2]))
        elif op[0] == "named":
            out.append(CLASS[op[1]](op[2], name=op[3], remapping=None))
        elif op[0] == "u":
            out.append(qandle.U(op[1], torch.from_numpy(U_MATRIX)))
        elif op[0] == "ctrl":
            out.append(qandle.Controlled(op[1], CLASS[op[2]](op[3], theta=theta[op[4]].clone(), remapping=None)))
        elif op[0] == "cz":
            out.append(qandle.CZ(op[1], op[2]))
        elif op[0] == "swap":
            out.append(qandle.SWAP(op[1], op[2]))
        elif op[0] == "reset":
            out.append(qandle.Reset(op[1]))
        else:
            out.append(CLASS[op[0]](op[1], theta=theta[op[2]].clone(), remapping=None))
    return out


def _structure(case):
    kind = case["kind"]
    if kind in ("forward", "train"):
        return _family(case["family"], case["n"], case["depth"])
    return {"reupload": _reupload, "amplitude": _sel, "gates": _gates}[kind](case["n"], case["depth"])


def _draws(case, seed):
    """Angles, inputs and loss weights of a single-circuit case (host tensors)."""
    gen = torch.Generator().manual_seed(seed)
    n, B, kind = case["n"], case["B"], case["kind"]
    ops, k = _structure(case)
    theta = torch.rand(k, generator=gen) * (2 * math.pi)
    if kind == "amplitude":
        x = torch.randn(B, case["features"], generator=gen)
    elif kind == "reupload":
        x = torch.rand(n, B, generator=gen) * math.pi
    else:
        x = torch.rand(B, n, generator=gen) * math.pi
    w = torch.randn(B, 2 ** n if kind == "amplitude" else n, generator=gen)
    return ops, theta, x, w


def _qconv(case, seed):
    gen = torch.Generator().manual_seed(seed)
    torch.manual_seed(seed)
    layer = qandle.QConv(case["c_in"], case["c_out"], kernel_size=case["k"], padding=1, qdepth=case["depth"])
    x = torch.rand(case["b"], case["c_in"], case["h"], case["w"], generator=gen)
    h, w = case["h"] + 3 - case["k"], case["w"] + 3 - case["k"]
    lw = torch.randn(case["b"], case["c_out"], h, w, generator=gen)
    return layer, x, lw


def _uneven(case, seed):
    """The mix's circuits with the seed's angles, inputs and loss weights."""
    ws = workloads.random_uneven(num_circuits=case["count"], n_hi=case["n_hi"], seed=case["mix"], build_layers=False)
    rng = np.random.default_rng(seed)
    lw = []
    for w in ws:
        w.gates = [g if g[0] == "cnot" else (g[0], g[1], float(np.float32(rng.uniform(0, 2 * math.pi)))) for g in w.gates]
        w.inputs["x"] = torch.from_numpy(rng.uniform(0, math.pi, (1, w.n)).astype(np.float32))
        lw.append(torch.from_numpy(rng.standard_normal((1, w.n)).astype(np.float32)))
    return ws, lw


def _requests(case, seed):
    """(n, B, depth) of the mix's requests and the seed's workloads."""
    rng = np.random.default_rng(case["mix"])
    gen = torch.Generator().manual_seed(seed)
    out = []
    for _ in range(case["count"]):
        n = 99
        while n > case["n_hi"]:
            n = 9 + int(rng.geometric(1 / 7))
        out.append(workloads.hardware_efficient(n, int(rng.integers(1, case["b_max"] + 1)), int(rng.integers(4, 13)), gen))
    return out


# ---------------------------------------------------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "qconv":
        layer, x, w = _qconv(case, seed)
        s["module"], s["x"], s["w"] = layer.to(DEV), x.to(DEV).requires_grad_(True), w.to(DEV)
        s["params"] = list(s["module"].parameters())
    elif kind == "uneven":
        ws, lw = _uneven(case, seed)
        ub = UnevenBatch.from_workloads(ws, DEV)
        ub.set_loss_weights(lw)
        ub.capture(backward=True)
        s["batch"] = ub
    elif kind == "serve":
        s["work"] = [(qandle.Circuit(w.layers, num_qubits=w.n).to(DEV), {"x": w.inputs["x"].to(DEV)})
                     for w in _requests(case, seed)]
        s["engine"] = None
    else:
        ops, theta, x, w = _draws(case, seed)
        n = case["n"]
        wires = list(range(n))
        if kind == "amplitude":
            layers = [qandle.AmplitudeEmbedding(name="x", qubits=wires, pad_with=0.0, normalize=True),
                      qandle.StronglyEntanglingLayer(qubits=wires, depth=case["depth"], remapping=None,
                                                     q_params=theta.reshape(case["depth"], n, 3)),
                      qandle.MeasureJointProbability()]
        else:
            layers = [] if kind == "reupload" else [qandle.AngleEmbedding(name="x", qubits=wires, rotation="rx")]
            layers += _layers(ops, theta) + [qandle.MeasureProbability()]
        s["module"] = qandle.Circuit(layers, num_qubits=n).to(DEV)
        s["params"] = [p for name, p in s["module"].named_parameters()
                       if not (kind == "reupload" and s["module"].get_submodule(name.rsplit(".", 1)[0]).named)]
        s["w"] = w.to(DEV)
        if kind == "reupload":
            s["inputs"] = {f"x{q}": x[q].to(DEV).requires_grad_(True) for q in range(n)}
        else:
            s["x"] = x.to(DEV).requires_grad_(kind != "forward")
    return s


def run(s):
    kind = s["kind"]
    if kind == "forward":
        with torch.no_grad():
            return s["module"](x=s["x"])
    if kind == "uneven":
        ub = s["batch"]
        ub.replay(backward=True)
        return ub.out, ub.grad_phi, ub.grad_x
    if kind == "serve":
        if s["engine"] is None:
            s["engine"] = serving.ServingEngine(DEV, cap_bytes=8e9, compiled_from_qubits=18)
        eng = s["engine"]
        eng.done = []
        reqs = [eng.prepare(serving.Request(i, c, kw)) for i, (c, kw) in enumerate(s["work"])]
        eng.serve(reqs)
        return [r.result for r in reqs]
    inputs = s.get("inputs") or {"x": s["x"]}
    for p in s["params"]:
        p.grad = None
    for v in inputs.values():
        v.grad = None
    out = s["module"](s["x"]) if kind == "qconv" else s["module"](**inputs)
    (out * s["w"]).sum().backward()
    gx = [v.grad for v in inputs.values()]
    return out.detach(), gx[0] if len(gx) == 1 else torch.stack(gx), _flat([p.grad for p in s["params"]])


def _flat(grads):
    return torch.stack(grads) if grads[0].dim() == 0 else torch.cat(grads)


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def _circuit_flops(ops, n, B):
    """Real operations of a state-vector run: 6 per amplitude for a rotation alone, 14 for a run of rotations on a
    qubit (one complex 2 x 2 product per pair); CNOT, CZ and SWAP move amplitudes only; 3 for a readout."""
    per, run_of = 0, {}

    def close(q):
        nonlocal per
        c = run_of.pop(q, 0)
        per += 0 if c == 0 else 6 if c == 1 else 14

    for op in ops:
        if op[0] in ("rx", "ry", "rz"):
            run_of[op[1]] = run_of.get(op[1], 0) + 1
        elif op[0] == "named":
            run_of[op[2]] = run_of.get(op[2], 0) + 1
        elif op[0] == "ctrl":
            close(op[1])
            close(op[3])
            per += 3
        elif op[0] in ("u", "reset"):
            close(op[1])
            per += 14
        else:
            close(op[1])
            close(op[2])
    for q in list(run_of):
        close(q)
    return (per + 3) * B * 2 ** n


def work(case):
    kind = case["kind"]
    if kind == "uneven":
        ws, _ = _uneven(case, 0)
        fl = sum(4 * _circuit_flops([("cnot", *g[1]) if g[0] == "cnot" else g for g in w.gates], w.n, 1) for w in ws)
        return {"bytes": sum(4 * 2 * sum(g[0] != "cnot" for g in w.gates) + 16 * w.n for w in ws), "flops": fl}
    if kind == "serve":
        ws = _requests(case, 0)
        fl = sum(_circuit_flops([("cnot", *g[1]) if g[0] == "cnot" else g for g in w.gates], w.n, w.B) for w in ws)
        return {"bytes": sum(8 * w.B * w.n + 4 * len(w.gates) for w in ws), "flops": fl}
    if kind == "qconv":
        n = max(math.ceil(math.log2(case["k"] ** 2 * case["c_in"])), math.ceil(math.log2(case["c_out"])), 1)
        px = case["b"] * (case["h"] + 3 - case["k"]) * (case["w"] + 3 - case["k"])
        ops, k = _sel(n, case["depth"])
        return {"bytes": 8 * case["b"] * case["c_in"] * case["h"] * case["w"] + 8 * px * case["c_out"] + 8 * k,
                "flops": 4 * _circuit_flops(ops, n, px)}
    ops, k = _structure(case)
    n, B = case["n"], case["B"]
    fl = _circuit_flops(ops, n, B)
    if kind == "forward":
        return {"bytes": 8 * B * n + 4 * k, "flops": fl}
    if kind == "amplitude":
        return {"bytes": 8 * B * 2 ** n + 8 * B * case["features"] + 8 * k, "flops": 4 * fl}
    return {"bytes": 16 * B * n + 8 * k, "flops": 4 * fl}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


# ---------------------------------------------------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------------------------------
def _rot(kind, phi):
    """((u00, u01), (u10, u11)) of a rotation by phi, each 0-d or (B, 1, 1), complex128."""
    c, s = torch.cos(phi / 2), torch.sin(phi / 2)
    if c.dim() == 1:
        c, s = c[:, None, None], s[:, None, None]
    z = torch.zeros_like(c)
    if kind == "rx":
        return (torch.complex(c, z), torch.complex(z, -s)), (torch.complex(z, -s), torch.complex(c, z))
    if kind == "ry":
        return (torch.complex(c, z), torch.complex(-s, z)), (torch.complex(s, z), torch.complex(c, z))
    return (torch.complex(c, -s), None), (None, torch.complex(c, s))


def _pair(psi, n, q, u, ctrl=None):
    v = psi.reshape(psi.shape[0], 2 ** q, 2, -1)
    a, b = v[:, :, 0], v[:, :, 1]
    r0 = u[0][0] * a + u[0][1] * b if u[0][1] is not None else u[0][0] * a
    r1 = u[1][0] * a + u[1][1] * b if u[1][0] is not None else u[1][1] * b
    out = torch.stack((r0, r1), 2).reshape(psi.shape)
    return out if ctrl is None else torch.where(_bit(n, ctrl), out, psi)


def _bit(n, q):
    return ((torch.arange(2 ** n, device=DEV) >> (n - 1 - q)) & 1).bool()


def _step(psi, n, op, theta, inputs):
    kind = op[0]
    if kind in ("rx", "ry", "rz"):
        return _pair(psi, n, op[1], _rot(kind, theta[op[2]]))
    if kind == "named":
        return _pair(psi, n, op[2], _rot(op[1], inputs[op[3]]))
    if kind == "ctrl":
        return _pair(psi, n, op[3], _rot(op[2], theta[op[4]]), ctrl=op[1])
    if kind == "u":
        m = torch.from_numpy(U_MATRIX).to(DEV).to(torch.complex128).T
        return _pair(psi, n, op[1], ((m[0, 0], m[0, 1]), (m[1, 0], m[1, 1])))
    if kind == "reset":
        v = psi.reshape(psi.shape[0], 2 ** op[1], 2, -1)
        a, b = v[:, :, 0], v[:, :, 1]
        norm = torch.sqrt(a.real ** 2 + a.imag ** 2 + b.real ** 2 + b.imag ** 2)
        a = a * (norm / (torch.sqrt(a.real ** 2 + a.imag ** 2) + 1e-7))
        return torch.stack((a, torch.zeros_like(a)), 2).reshape(psi.shape)
    idx = torch.arange(2 ** n, device=DEV)
    x, y = 1 << (n - 1 - op[1]), 1 << (n - 1 - op[2])
    if kind == "cnot":
        return psi[:, torch.where((idx & x) != 0, idx ^ y, idx)]
    if kind == "swap":
        return psi[:, torch.where(((idx & x) != 0) != ((idx & y) != 0), idx ^ (x | y), idx)]
    return torch.where(((idx & x) != 0) & ((idx & y) != 0), -psi, psi)  # cz


def _zero(n, B):
    psi = torch.zeros(B, 2 ** n, dtype=torch.complex128, device=DEV)
    psi[:, 0] = 1
    return psi


def _simulate(n, ops, theta, x=None, inputs=None, psi=None, joint=False):
    """P(qubit = 0) (or |psi|^2) of the embedded state after ``ops``."""
    if psi is None:
        B = x.shape[0] if x is not None else next(iter(inputs.values())).shape[0]
        psi = _zero(n, B)
    if x is not None:
        for q in range(n):
            psi = _pair(psi, n, q, _rot("rx", x[:, q]))
    for op in ops:
        psi = _step(psi, n, op, theta, inputs)
    p = psi.real ** 2 + psi.imag ** 2
    if joint:
        return p
    return torch.stack([p.reshape(p.shape[0], 2 ** q, 2, -1)[:, :, 0].sum((1, 2)) for q in range(n)], 1)


def _chunk(n, count, grad):
    """Samples at a time: with gradients every operator's input state stays."""
    return max(1, int(24e9 // (16 * 2 ** n * (1.2 * count + 8 if grad else 8))))


def _workload_exact(w, lw=None):
    theta = torch.tensor([g[2] for g in w.gates if g[0] != "cnot"], dtype=torch.float64, device=DEV)
    ops, k = [], 0
    for g in w.gates:
        if g[0] == "cnot":
            ops.append(("cnot", *g[1]))
        else:
            ops.append((g[0], g[1], k))
            k += 1
    x = w.inputs["x"].to(DEV).double()
    if lw is None:
        with torch.no_grad():
            return _simulate(w.n, ops, theta, x)
    theta.requires_grad_(True)
    x.requires_grad_(True)
    p = _simulate(w.n, ops, theta, x)
    (p * lw.to(DEV).double()).sum().backward()
    return p.detach(), theta.grad, x.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "uneven":
        if case["count"] > 64:  # some minutes of small launches: the drawn cases of fewer circuits have a value
            return None
        ws, lw = _uneven(case, seed)
        got = [_workload_exact(w, v) for w, v in zip(ws, lw)]
        return tuple(torch.cat([g[i].reshape(-1) for g in got]) for i in range(3))
    if kind == "serve":
        return [_workload_exact(w) for w in _requests(case, seed)]
    if kind == "qconv":
        layer, x, w = _qconv(case, seed)
        ops, _ = _sel(layer.qubits, case["depth"])
        raw = torch.stack([p.detach().reshape(()) for p in layer.parameters()]).to(DEV).double().requires_grad_(True)
        x = x.to(DEV).double().requires_grad_(True)
        cols = torch.nn.functional.unfold(x, case["k"], padding=1)
        rows = cols.transpose(1, 2).reshape(-1, cols.shape[1]) + 0.001
        psi = torch.nn.functional.pad(rows, (0, 2 ** layer.qubits - rows.shape[1])).to(torch.complex128)
        p = _simulate(layer.qubits, ops, math.pi * torch.tanh(raw), psi=psi, joint=True)
        img = p.reshape(w.shape[0], w.shape[2], w.shape[3], -1).permute(0, 3, 1, 2)
        out = img[:, : case["c_out"]] * (case["c_out"] / 2)
        (out * w.to(DEV).double()).sum().backward()
        return out.detach(), x.grad, raw.grad
    ops, theta, x, w = _draws(case, seed)
    n = case["n"]
    theta, x, w = theta.to(DEV).double(), x.to(DEV).double(), w.to(DEV).double()
    if kind == "forward":
        with torch.no_grad():
            p = torch.cat([_simulate(n, ops, theta, xs) for xs in x.split(_chunk(n, 0, False))])
        return p.squeeze(0) if case["B"] == 1 else p
    theta.requires_grad_(True)
    x.requires_grad_(True)
    samples = _chunk(n, len(ops) + n, True)
    outs = []
    for lo in range(0, case["B"], samples):
        ws = w[lo:lo + samples]
        if kind == "reupload":
            xs = x[:, lo:lo + samples]
            p = _simulate(n, ops, theta, inputs={f"x{q}": xs[q] for q in range(n)})
        elif kind == "amplitude":
            v = torch.nn.functional.pad(x[lo:lo + samples], (0, 2 ** n - case["features"]))
            p = _simulate(n, ops, theta, psi=torch.nn.functional.normalize(v, dim=1).to(torch.complex128), joint=True)
        else:
            p = _simulate(n, ops, theta, x[lo:lo + samples])
        (p * ws).sum().backward()
        outs.append(p.detach())
    p = torch.cat(outs)
    return p.squeeze(0) if case["B"] == 1 and kind != "amplitude" else p, x.grad, theta.grad
