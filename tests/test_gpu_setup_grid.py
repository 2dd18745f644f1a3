"""qs_setup with more blocks than one row of a launch's grid takes (a block per table and sample)."""
import ctypes

import pytest
import torch

from qandle_amd._engine import givens as GV
from qandle_amd._engine import lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,ntables", [(5, 3), (2 ** 20 + 7, 65)])
def test_tables_of_many_samples(device, B, ntables):
    """Tables of one entry: the number e^{-i phi_b / 2} of an RZ, the same in every table."""
    half = torch.rand(B, device=device, generator=torch.Generator(device=device).manual_seed(0)) * 3
    cs = torch.stack((torch.cos(half), torch.sin(half)), 1).contiguous()
    words = []
    for t in range(ntables):
        words += [2 * B * t, 1, 0, 1, GV.ZNUM | L.FACTOR_PER_SAMPLE, 0, 0]
    index = torch.tensor(words + [7 * t for t in range(ntables)], dtype=torch.int32, device=device)
    out = torch.full((ntables, B, 2), float("nan"), device=device)
    a = L.SetupArgs()
    a.B, a.n, a.cs, a.gtab, a.ltab, a.words = B, 1, L.ptr(cs), L.ptr(out), L.ptr(out), L.ptr(index)
    a.twords, a.tables, a.nstables = L.ptr(index), L.ptr(index) + 4 * len(words), ntables
    L.check(L.load().qs_setup(ctypes.byref(a), L.stream_of(cs)), "qs_setup")
    want = cs * torch.tensor([1.0, -1.0], device=device)
    assert all(torch.equal(out[t], want) for t in range(ntables))
