"""Adjoint backward of a fused program, behind one torch.autograd.Function.

Forward: the fused passes, keeping the final state and a copy of the state
every ``checkpoint_gates`` gates (at pass boundaries).

Backward (reverse sweep over the same passes, ``qs_adjoint_pass``):

* co-state seed: lambda = 2 psi * sum_q w_q [bit n-1-q = 0] for a
  MeasureProbability output (w = dL/dP), or dL/dpsi for a state output;
  when the compiled kernels fold trailing CNOTs into the readout, psi is the
  state before them and the measured bit is the parity of its readout mask;
* per pass, in reverse: for every gate, 1/2 Im<lambda|P|psi> at its output,
  then psi <- U^dag psi, lambda <- U^dag lambda;
* where a checkpoint exists, psi is reset to it, which bounds the float32
  drift of un-applying gates on a deep circuit;
* AngleEmbedding inputs: dL/dx_j = 1/2 Im<lambda_0|P_j|psi_0> (the embedded
  factors commute, so every column comes from the one final pair);
* an initial state that needs a gradient gets lambda_0.

Gradients of remapped parameters flow through torch (``remap(theta)`` is
computed outside the Function).
"""
from __future__ import annotations

import ctypes
import dataclasses
import typing

import numpy as np
import torch

from .. import config
from . import fused
from . import lib as L


# When set to a list, the backward sweep appends (start, end, algorithmic bytes)
# for every adjoint kernel launch: HIP events recorded on the launch stream.
# Measurement only (the benchmark's roofline of the adjoint kernels).
launch_events = None


def checkpoint_after(prog, pl, every_gates: int):
    """Pass indices after which the forward state is stored."""
    out = set()
    done = 0
    next_mark = every_gates
    for i, p in enumerate(pl.passes[:-1]):
        done += len(p.gates)
        if every_gates > 0 and done >= next_mark:
            out.add(i)
            while next_mark <= done:
                next_mark += every_gates
    return out


def default_checkpoint_gates(n: int) -> int:
    """CHECKPOINT_LAYERS layers of (RX, RY, RZ per qubit + a CNOT per qubit)."""
    return int(config.CHECKPOINT_LAYERS) * 4 * n


class FusedCircuitFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, prog, R, TB, cm, B, batched, names, phi_param, embed_x, state, *named_vals):
        named = dict(zip(names, [v.detach() for v in named_vals]))
        inp = fused.Inputs(B, batched, phi_param.device, phi_param.detach(), named,
                           None if embed_x is None else embed_x.detach(),
                           None if state is None else state.detach())
        jit_on = fused.use_jit(prog.n, R, TB)
        fold = fused.folds(prog, jit_on)
        pl = fused.get_plan(prog, R, TB, cm, fold)
        every = config.CHECKPOINT_GATES if getattr(config, "CHECKPOINT_GATES", None) else default_checkpoint_gates(prog.n)
        ckpts = dict.fromkeys(checkpoint_after(prog, pl, every))  # pass outputs kept for the sweep
        psi, probs, cs = fused._execute(prog, inp, None, None, R, TB, cm=cm, want_state=True, marks=ckpts,
                                        specialise=jit_on, fold=fold)
        ctx.prog, ctx.R, ctx.TB, ctx.cm, ctx.B, ctx.names = prog, R, TB, cm, B, names
        ctx.jit, ctx.fold = jit_on, fold
        ctx.ck_index = sorted(ckpts)
        ctx.named_shapes = [v.shape for v in named_vals]
        ctx.embed_shape = None if embed_x is None else embed_x.shape
        ctx.state_shape = None if state is None else state.shape
        ctx.save_for_backward(psi, cs, *[ckpts[i] for i in ctx.ck_index])
        if prog.measure:
            return probs
        return psi

    @staticmethod
    def backward(ctx, gout):
        prog, R, TB, B = ctx.prog, ctx.R, ctx.TB, ctx.B
        saved = ctx.saved_tensors
        psi_final, cs = saved[0], saved[1]
        ckpts = dict(zip(ctx.ck_index, saved[2:]))
        n = prog.n
        lib = L.load()
        st = L.stream_of(psi_final)
        # the compiled steps read psi from psi_src and write psi: the first reads the saved final
        # state and each reset reads its checkpoint, with no copies; the interpreting steps work in place
        psi = torch.empty_like(psi_final) if ctx.jit else psi_final.clone()
        psi_src = psi_final
        lam = torch.empty_like(psi)
        seed = None
        if prog.measure:
            # the first adjoint pass builds lambda from psi and w = dL/dP while loading
            seed = gout.to(torch.float32).contiguous()
        else:
            lam.copy_(gout.to(torch.complex64).resolve_conj())
        embed = prog.init[0] == "embed" and ctx.needs_input_grad[8]
        opts = getattr(config, "SPECIALISE_ADJOINT_OPTIONS", None)
        call = prog.kept(("adjoint_call", R, TB, ctx.cm.key(), B, psi.device.index, ctx.jit, ctx.fold, embed,
                          seed is not None, tuple(sorted(opts.items())) if opts else ()),
                         lambda: _adjoint_call(prog, R, TB, ctx.cm, B, psi.device, ctx.jit, ctx.fold, embed,
                                               seed is not None))
        call.tables.use(st, psi.device)
        ws, kern, NS, ntiles = call.ws, call.kern, call.NS, call.ntiles
        # the unitaries, their generators and U^dagger operands (step by step), from the forward's half angles,
        # and the sweep's partials
        n_u, n_q, n_l, n_g = call.sizes
        work = torch.empty(n_u + n_q + n_l + n_g, dtype=torch.float32, device=psi.device)
        utab = L.ptr(work)
        qtab, ltab, gpart = utab + 4 * n_u, utab + 4 * (n_u + n_q), utab + 4 * (n_u + n_q + n_l)
        args = call.setup.fill(B, L.ptr(cs), utab, ltab, qtab=qtab)
        events = launch_events
        npass = len(call.pl.passes)
        seed_ptr = None if seed is None else L.ptr(seed)
        if kern is not None and events is None:
            sources = (ctypes.c_void_p * len(ws.passes))()
            sources[0] = L.ptr(psi_src)
            for i in ckpts:  # the step after the one that undoes pass i + 1 starts from pass i's kept output
                sources[npass - 1 - i] = L.ptr(ckpts[i])
            block = L.AdjointCall(L.ptr(psi), L.ptr(lam), utab, qtab, L.ptr(cs), gpart, seed_ptr, ltab, None, B, NS, ntiles)
            L.check(lib.qs_run_adjoint(ctypes.byref(args), len(ws.passes), call.functions, call.grid, kern.block, sources,
                                       ctypes.byref(block), st), "qs_run_adjoint")
        else:
            L.check(lib.qs_setup(ctypes.byref(args), st), "qs_setup")
            for k, (w, nsub, lpos) in enumerate(ws.passes):
                seeded = seed_ptr if k == 0 else None
                if events is not None:
                    ev = (torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
                    ev[0].record(torch.cuda.current_stream(psi.device))
                if kern is not None:
                    kern.launch(k, L.ptr(psi), L.ptr(lam), utab, qtab, L.ptr(cs), gpart, seeded, B, NS, ntiles, st, ltab,
                                L.ptr(psi_src))
                    psi_src = psi
                else:
                    L.check(
                        lib.qs_adjoint_pass(
                            L.ptr(psi), L.ptr(lam), B, n, R, TB,
                            lpos.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), L.ptr(w), nsub,
                            L.ptr(cs), utab, qtab, gpart, call.rows, seeded, st,
                        ),
                        "qs_adjoint_pass",
                    )
                if events is not None:
                    ev[1].record(torch.cuda.current_stream(psi.device))
                    # psi and lambda are read and written once per step; a seeded step reads psi only
                    events.append((ev[0], ev[1], B * (2 ** n) * (24 if seeded is not None else 32)))
                i = npass - 1 - k  # forward pass this step undid
                if k < call.nmain and (i - 1) in ckpts:
                    if kern is not None:
                        psi_src = ckpts[i - 1]
                    else:
                        psi.copy_(ckpts[i - 1])
        # every gradient the call returns, from the partials, in one launch
        need_param = bool(ctx.needs_input_grad[7])
        named = tuple((name, len(shape) > 0) for k, (name, shape) in enumerate(zip(ctx.names, ctx.named_shapes))
                      if ctx.needs_input_grad[10 + k])
        batched_x = embed and len(ctx.embed_shape) > 1
        route = gradient_route(prog, B, psi.device, need_param, named, embed, batched_x)
        route.tables.use(st, psi.device)
        grads = torch.empty(route.size, dtype=torch.float32, device=psi.device)
        if route.ngroups:
            base = L.ptr(route.index)
            L.check(lib.qs_gradients(L.ptr(grads), gpart, base + route.first, base + route.rows, base,
                                     route.ngroups, B, NS, slots_per_sample(B, n, R, TB), st), "qs_gradients")
        # tensors of their own on the buffer (.data: with version counters of their own, so that one
        # changed in place leaves what autograd saved of another valid)
        g_param = grads[:len(prog.param_slots)].data if need_param else None
        g_named = []
        for k, shape in enumerate(ctx.named_shapes):
            lo = route.named.get(ctx.names[k])
            g_named.append(None if lo is None else grads[lo].data if len(shape) == 0
                           else grads[lo:lo + B].data.reshape(shape))
        g_embed = None
        if embed:
            lo = route.embed
            g_embed = grads[lo:lo + len(prog.init[2])].data if not batched_x else grads[lo:].data.reshape(ctx.embed_shape)
        g_state = None
        if ctx.needs_input_grad[9] and prog.init[0] != "embed":
            shp = ctx.state_shape
            g_state = lam.sum(0) if len(shp) == 1 else (lam if lam.shape == shp else lam.sum(0, keepdim=True))
        return (None, None, None, None, None, None, None, g_param, g_embed, g_state, *g_named)


@dataclasses.dataclass
class AdjointCall:
    """The part of an adjoint sweep that its calls share: plan, words, kernels, table
    sizes and the launch list (for qs_run_adjoint)."""

    pl: typing.Any
    ws: typing.Any
    nmain: int
    kern: typing.Any
    setup: typing.Any
    sizes: tuple              # floats of utab, qtab, ltab, the gradient partials
    rows: int
    ntiles: int
    NS: int
    tables: typing.Any
    functions: typing.Any = None
    grid: typing.Any = None


def _adjoint_call(prog, R, TB, cm, B, device, jit_on, fold, embed, seeded) -> AdjointCall:
    n = prog.n
    rows = len(fused.rotation_rows(prog)) + (len(prog.init[2]) if embed else 0)
    part = L.work_floats(L.load().qs_adjoint_work_bytes(B, n, R, TB, rows), "qs_adjoint_work_bytes")
    pl = fused.get_plan(prog, R, TB, cm, fold)
    ws, nmain = fused.adjoint_words(prog, pl, B, device, embed, cm)
    ntiles, NS = adjoint_geometry(B, n, R, TB)
    kern = specialised_adjoint(prog, pl, ws, B, embed, seeded, fold) if jit_on else None
    plan = fused.setup_plan(prog, ws, None if kern is None else kern.lane_index, B, device, dagger=True)
    call = AdjointCall(pl, ws, nmain, kern, plan, (max(plan.nu, 1) * 8, max(plan.nq, 1) * 8, max(plan.nlane, 16),
                                                   max(part, 1)), rows, ntiles, NS,
                       fused.Resident([*plan.keep, *([w for w, _, _ in ws.passes] if kern is None else [])]))
    if kern is not None:
        count = len(ws.passes)
        call.functions = (ctypes.c_void_p * count)(*[f.value for f in kern.funcs])
        call.grid = (ctypes.c_uint * count)(*[kern.grid(i, ntiles) for i in range(count)])
    return call


@dataclasses.dataclass
class GradientRoute:
    """qs_gradients' index arrays for one set of wanted gradients, in one device
    tensor (places first; ``first`` and ``rows`` are byte offsets into it), and
    where each gradient lies in the launch's output: the angles from 0, every
    named input, the embedded features."""

    index: torch.Tensor
    first: int
    rows: int
    ngroups: int
    size: int
    named: dict
    embed: int
    tables: typing.Any


def gradient_route(prog, B, device, need_param, named, embed, batched_x) -> GradientRoute:
    """Route of the gradient rows to the wanted gradients, kept with the program.
    ``named``: (name, whether it has an entry per sample) of the wanted named
    inputs; ``embed`` the embedded features (rows after the rotations'),
    ``batched_x``: as (B, d), else summed over the batch."""
    return prog.kept(("grad_route", B, device.index, need_param, named, embed, batched_x),
                     lambda: _gradient_route(prog, B, device, need_param, named, embed, batched_x))


def _gradient_route(prog, B, device, need_param, named, embed, batched_x) -> GradientRoute:
    rows = fused.rotation_rows(prog)
    by_slot, by_name = {}, {}
    for gi, g in enumerate(prog.gates):
        if g.kind == 4:  # CNOT
            continue
        sl = prog.slots[g.slot]
        if sl.kind == "param":
            by_slot.setdefault(g.slot, []).append(rows[gi])
        elif sl.kind == "named":
            by_name.setdefault(sl.name, []).append(rows[gi])
    groups, size, where = [], 0, {}  # (rows, first output, stride)
    if need_param:
        groups += [(by_slot.get(s_, []), i, 0) for i, s_ in enumerate(prog.param_slots)]
        size = len(prog.param_slots)
    for name, per_sample in named:
        groups.append((by_name.get(name, []), size, 1 if per_sample else 0))
        where[name] = size
        size += B if per_sample else 1
    at = size
    if embed:
        d = len(prog.init[2])
        groups += [([len(rows) + j], at + j, d if batched_x else 0) for j in range(d)]
        size += d * B if batched_x else d
    first = np.cumsum([0] + [len(g[0]) for g in groups])
    flat = [r for g in groups for r in g[0]]
    place = np.asarray([v for g in groups for v in g[1:]], dtype=np.int64)
    words = np.concatenate([place.view(np.int32), np.asarray(list(first) + flat, dtype=np.int32)])
    pad = np.zeros(len(words) % 2, dtype=np.int32)
    index = L.upload(np.concatenate([words, pad]).view(np.int64), torch.int64, device)
    return GradientRoute(index, 8 * len(place), 8 * len(place) + 4 * len(first), len(groups), size, where, at,
                         fused.Resident([index]))


def slots_per_sample(B: int, n: int, R: int, TB: int) -> int:
    """Reduction slots per sample of a gradient row (adjoint_geometry)."""
    K = R + TB
    seglog = (n - R) if n < K else TB
    wlog = min(seglog, 6)
    return 1 << (seglog - wlog) if n < K else (1 << (n - K)) << (TB - wlog)


def adjoint_geometry(B: int, n: int, R: int, TB: int):
    """(tiles, reduction slots per gradient row) of an adjoint pass, as the
    library's adjoint kernels and qs_adjoint_finish lay them out."""
    K = R + TB
    multi = n < K
    seglog = (n - R) if multi else TB
    wlog = min(seglog, 6)
    ntiles = ((B + (1 << (K - n)) - 1) >> (K - n)) if multi else (B << (n - K))
    return ntiles, ntiles * (1 << (TB - wlog))


def specialised_adjoint(prog, pl, ws, B, embed, seeded, fold=False):
    """Run-time compiled kernels of this plan's adjoint sweep (cached on the
    program); with ``fold`` the seed reads the readout masks of the folded
    trailing CNOTs (fused.readout_fold)."""
    from . import jit

    opts = getattr(config, "SPECIALISE_ADJOINT_OPTIONS", {}) or {}

    def make():
        masks = fused.readout_fold(prog)[1] if fold else None
        return jit.AdjointKernels(ws.host_passes(), prog.n, pl.R, pl.TB, seeded, readout=masks, **opts)

    return prog.kept(("jit_adj", id(pl), B, embed, seeded, fold, tuple(sorted(opts.items()))), make)


def run_with_grad(prog, inp, R, TB, cm=None):
    names = list(inp.named)
    vals = [inp.named[k] for k in names]
    out = FusedCircuitFn.apply(prog, R, TB, cm or fused.GRAD_COST, inp.B, inp.batched, names, inp.phi_param,
                               inp.embed_x, inp.state, *vals)
    if prog.measure:
        return None, out
    return out, None
