"""Fused unitaries of the compiled forward passes as real rotations between diagonals.

A fused unitary is a product of rotations, so U = a D R G with the diagonals
G = diag(1, g) and D = diag(1, w), a number a, and the real matrix R =
[[1, -t], [t, 1]] or, past 45 degrees, [[t, -1], [1, t]], 0 <= t <= 1 (a scaled
rotation; qs_setup picks the form, a uniform branch of the kernel).  On the
vector ALU that is 4 fused multiply-adds per amplitude pair against 16 for a
complex 2x2 product, and the diagonals of neighbouring unitaries merge: what
is pending on the registers that the next unitary mixes is one complex factor
per register, a table multiplication.  A diagonal waits (``carry``) while its
bit is not a register, past CNOTs that it controls, past sub-passes and
passes, until its bit is rotated again; one that is never rotated again before
a measurement is dropped.  The numbers a (R grows an amplitude by at most
sqrt(2)) join a table once NUMBERS of them wait; the last ones start the
generated state.

The matrix cores do not help here: gfx950 runs v_mfma_f32_4x4x1f32 on the
vector pipes (measured: 153 TFLOP/s of it alone, 127 of vector FMAs alone, and
the two interleaved take 1.3 times the sum of their times), so the fewest
operations win.

:class:`Schedule` turns a program's decoded passes into steps for the code
generator (jit) and the list of records (one per unitary) and tables (one per
diagonal product) that qs_setup fills.
"""
from __future__ import annotations

import dataclasses

from . import lib as L
from . import planner as PL

# kinds of a diagonal factor (include/qandle_sv.h), the value where its parity is 1 (it is 1
# where the parity is 0): g and w of a unitary, e^{i phi} of an RZ; and of the numbers: a
# unitary's a, an RZ's e^{-i phi / 2}
G, W, ZW, NUM, ZNUM = 0, 1, 2, 3, 4
RECORD = 8    # floats per unitary: t, the form, g, w, a
# Numbers that wait before they are applied.  They are looked at where a segment starts, so up to
# NUMBERS - 1 + R unitaries may pass: amplitudes grow by at most 2^34 (R <= 5)
NUMBERS = 64


@dataclasses.dataclass(frozen=True)
class Factor:
    kind: int
    ref: int      # utab index of the unitary, cs index of an RZ
    ps: bool      # per sample


def parity(x: int) -> int:
    return bin(x).count("1") & 1


class Registers:
    """Register renaming of a sub-pass (a linear map of the index bits) and the
    diagonals pending on the physical registers: (factor, mask), whose value at
    physical register k is the factor's value at parity(mask & k)."""

    def __init__(self, R: int):
        self.R = R
        self.phys = list(range(1 << R))
        self.pending: list = []

    def mask_of(self, r: int) -> int:
        """The mask whose parity is logical bit r of the register a physical index holds."""
        d = [self.phys[1 << s] for s in range(self.R)]
        return next(m for m in range(1, 1 << self.R) if all(parity(m & d[s]) == (s == r) for s in range(self.R)))

    def moves(self, mask: int, r: int) -> bool:
        """Whether flipping logical bit r flips the parity of ``mask``."""
        return bool(parity(mask & self.phys[1 << r]))

    def pairs(self, r: int):
        return [(self.phys[j], self.phys[j | (1 << r)]) for j in range(1 << self.R) if not (j >> r) & 1]

    def rename(self, tgt: int, ctl: int):
        for j in range(1 << self.R):
            if (j >> ctl) & 1 and not (j >> tgt) & 1:
                k = j | (1 << tgt)
                self.phys[j], self.phys[k] = self.phys[k], self.phys[j]


class Schedule:
    """Steps of every sub-pass of a forward program's passes.

    ``passes``: decoded sub-passes (planner.decode_pass) per pass; ``multi``:
    tiles of several samples (their per-sample unitaries stay complex products,
    as neighbouring lanes may hold different ones); ``generated``: the first
    pass makes its state, starting from the number of table 0, else that
    number joins the first table; ``exact_after``: passes whose stored state
    must hold every diagonal and number (checkpoints, a returned state).
    Steps of a sub-pass, in order:

    * ("table", index, registers): those registers times their table entries (1 for the others)
    * ("rot", record, ps, pairs), ("gen", utab index, pairs), ("swap", position, pairs)
    * ("thread", factors): every register times the product of the factors'
      values at the thread's own bits, [(factor, position)]
    """

    def __init__(self, passes, R: int, multi: bool, generated: bool, exact_after=()):
        self.R, self.multi = R, multi
        self.records: dict = {}   # (utab index, ps) -> record number
        self.tables: list = [[]]  # [(factor, mask)] per table; 0: the starting number of a generated state
        self.numbers: list = []   # numbers not applied yet
        self.steps: list = []     # [pass][sub-pass] -> (steps, phys, phases left to the thread loop)
        if exact_after and len(passes) - 1 not in exact_after:
            raise ValueError("numbers after the last exact state have no place to go")
        carry: dict = {}          # position -> [factor]
        for i, subs in enumerate(passes):
            out = []
            for k, sub in enumerate(subs):
                out.append(self._sub_pass(sub, carry, k == len(subs) - 1 and i in exact_after))
            self.steps.append(out)
        if generated:
            self.tables[0] = [(f, 0) for f in self.numbers]
        elif self.numbers:
            # an input state: with the first table, or one of their own
            steps = self.steps[0][0][0]
            if not steps or steps[0][0] != "table":
                self.tables.append([])
                steps.insert(0, ("table", len(self.tables) - 1, ()))
            kind, t, _regs = steps[0]
            self.tables[t] += [(f, 0) for f in self.numbers]
            steps[0] = (kind, t, tuple(range(1 << R)))
        self.start = bool(self.tables[0])

    def record(self, u: int, ps: bool) -> int:
        return self.records.setdefault((u, ps), len(self.records))

    def _table(self, steps, factors):
        if not factors:
            return
        for f, _ in factors:
            if f.kind in (G, W, NUM):
                self.record(f.ref, f.ps)
        numbers = [x for x in factors if x[0].kind in (NUM, ZNUM)]
        masked = [x for x in factors if x[0].kind not in (NUM, ZNUM)]
        for k in range(0, max(len(masked), 1), L.SETUP_MAX_FACTORS):  # as many as qs_setup multiplies into a table
            part = masked[k:k + L.SETUP_MAX_FACTORS]
            regs = tuple(j for j in range(1 << self.R) if numbers or any(parity(m & j) for _, m in part))
            steps.append(("table", len(self.tables), regs))
            self.tables.append(part + numbers)
            numbers = []

    def _flush(self, regs: Registers, steps, hit, extra=()):
        """A table of the pending diagonals that ``hit`` picks, with ``extra``."""
        take = [(f, m) for f, m in regs.pending if hit(m)]
        regs.pending = [(f, m) for f, m in regs.pending if not hit(m)]
        self._table(steps, take + list(extra))

    def _sub_pass(self, sub, carry, exact):
        regs, steps = Registers(self.R), []
        for r in range(self.R):
            regs.pending += [(f, 1 << r) for f in carry.pop(sub.GP[r], [])]
        for bits, cnots in sub.segments:
            real = [(r, u, ps) for r, u, ps in bits if not (ps and self.multi)]
            gen = [(r, u) for r, u, ps in bits if ps and self.multi]
            mixed = [r for r, _u, _ps in real] + [r for r, _u in gen]
            extra = [(Factor(G, u, ps), regs.mask_of(r)) for r, u, ps in real]
            if len(self.numbers) >= NUMBERS and real:
                extra += [(f, 0) for f in self.numbers]
                self.numbers = []
            self._flush(regs, steps, lambda m: any(regs.moves(m, r) for r in mixed), extra)
            for r, u, ps in real:
                steps.append(("rot", self.record(u, ps), ps, regs.pairs(r)))
                regs.pending.append((Factor(W, u, ps), regs.mask_of(r)))
                self.numbers.append(Factor(NUM, u, ps))
            for r, u in gen:
                steps.append(("gen", u, regs.pairs(r)))
            for uniform, tgt, ctl in cnots:
                if uniform:
                    self._flush(regs, steps, lambda m: regs.moves(m, tgt))
                    steps.append(("swap", ctl, regs.pairs(tgt)))
                else:
                    regs.rename(tgt, ctl)
        # RZ gates on bits outside the registers: diagonals of those bits
        left = []
        for pos, ci, fl in sub.phases:
            if fl & PL.SEG_NOUNAPPLY:
                continue
            if fl & PL.SEG_PER_SAMPLE and self.multi:
                left.append((pos, ci, fl))
            else:
                ps = bool(fl & PL.SEG_PER_SAMPLE)
                carry.setdefault(pos, []).append(Factor(ZW, ci, ps))
                self.numbers.append(Factor(ZNUM, ci, ps))
        masks = {regs.mask_of(r): sub.GP[r] for r in range(self.R)}
        if exact:
            self._flush(regs, steps, lambda m: True, [(f, 0) for f in self.numbers])
            self.numbers = []
            rest = [(f, pos) for pos, fs in carry.items() for f in fs]
            carry.clear()
            if rest:
                for f, _ in rest:
                    if f.kind != ZW:
                        self.record(f.ref, f.ps)
                steps.append(("thread", rest))
        else:
            self._flush(regs, steps, lambda m: m not in masks)  # a diagonal of several bits' parity cannot wait
        for f, m in regs.pending:
            carry.setdefault(masks[m], []).append(f)
        return steps, regs.phys, left

    def layout(self, B: int):
        """(float offset of every record, of every table, total floats) of the filled
        buffer: records first, per-sample ones B times."""
        rec, at = [], 0
        for (_u, ps) in self.records:
            rec.append(at)
            at += RECORD * (B if ps else 1)
        tab = []
        for factors in self.tables:
            tab.append(at)
            at += (2 << self.R) * (B if any(f.ps for f, _ in factors) else 1)
        return rec, tab, at
