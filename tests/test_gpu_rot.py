"""qs_rot_angle / qs_rot_backward (a rotation and its gradients straight from the angle)
against float64: every bit of small and chunk-sized states (the backward sums chunks of 2^11
pairs), control masks, per-sample and strided angles, states that are 8- but not 16-byte
aligned, either gradient alone, and an angle overwritten between forward and backward.

Bars: states within 4 ulp of their largest amplitude (two products and a sum per component);
gradients within 2^-20 of the sum of the magnitudes they add (float sums of at most 2^12 terms
per thread and block, double after that)."""
import numpy as np
import pytest
import torch

from oracle import fp64
from qandle_amd._engine import plain

pytestmark = pytest.mark.gpu
PAULI = ("x", "y", "z")


def _aligned_to_8(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    flat.copy_(t.reshape(-1))
    out = flat.view(t.shape)
    assert out.data_ptr() % 16 == 8
    return out


def _check(device, n, B, bit, kind, cmask, per_sample, misaligned):
    gen = torch.Generator().manual_seed(1000 * n + 10 * bit + kind + B)
    psi = torch.randn(B, 2 ** n, dtype=torch.complex64, generator=gen)
    g = torch.randn(B, 2 ** n, dtype=torch.complex64, generator=gen)
    wide = torch.rand(B, 3, generator=gen) * 6
    phi = wide[:, 1] if per_sample else wide[0, 1]
    on = np.ones(2 ** n, dtype=bool) if cmask == 0 else (np.arange(2 ** n) & cmask) == cmask
    U = fp64.rot_matrix(PAULI[kind], phi.double().numpy())
    p0 = psi.numpy().astype(np.complex128)
    g0 = g.numpy().astype(np.complex128)
    ref = np.where(on, fp64.apply_1q(p0, n, n - 1 - bit, U), p0)
    Ud = np.conj(np.swapaxes(U, -1, -2))
    gref = np.where(on, fp64.apply_1q(g0, n, n - 1 - bit, Ud), g0)
    terms = np.conj(g0) * fp64.apply_1q(ref, n, n - 1 - bit, fp64.PAULI[PAULI[kind]]) * on
    aref, mag = 0.5 * terms.imag.sum(1), 0.5 * np.abs(terms).sum(1)
    if not per_sample:
        aref, mag = aref.sum(), mag.sum()
    put = (lambda t: _aligned_to_8(t.to(device))) if misaligned else (lambda t: t.to(device))
    for want_state, want_phi in ((True, True), (True, False), (False, True)):
        st = put(psi).requires_grad_(want_state)
        base = wide.to(device)
        ph = (base[:, 1] if per_sample else base[0, 1]).detach().requires_grad_(want_phi)
        if cmask:
            out = plain.ControlledRotFn.apply(st, ph, n, bit, kind, cmask)
        else:
            out = plain.RotFn.apply(st, ph, n, bit, kind)
        base.zero_()  # the angle's memory changes after the forward
        assert np.abs(out.detach().cpu().numpy() - ref).max() <= 4 * 2.0 ** -24 * np.abs(ref).max() * 2
        out.backward(put(g))
        if want_state:
            assert np.abs(st.grad.cpu().numpy() - gref).max() <= 4 * 2.0 ** -24 * np.abs(gref).max() * 2
        if want_phi:
            err = np.abs(ph.grad.cpu().numpy() - aref)
            assert (err <= 2.0 ** -20 * mag).all(), (err, mag)


@pytest.mark.parametrize("n,B", [(1, 1), (1, 5), (2, 3), (3, 1), (5, 7)])
@pytest.mark.parametrize("misaligned", [False, True])
def test_small_states_every_bit(device, n, B, misaligned):
    for bit in range(n):
        for kind in range(3):
            for per_sample in (False, True):
                _check(device, n, B, bit, kind, 0, per_sample, misaligned)
                if n > 1:
                    _check(device, n, B, bit, kind, 1 << ((bit + 1) % n), per_sample, misaligned)


@pytest.mark.parametrize("n,B,bit", [(12, 2, 0), (12, 2, 11), (13, 3, 0), (13, 3, 1), (13, 3, 12), (14, 1, 5)])
def test_chunks(device, n, B, bit):
    for kind in range(3):
        _check(device, n, B, bit, kind, 0, kind == 1, False)
        _check(device, n, B, bit, kind, (1 << ((bit + 3) % n)) | (1 << ((bit + 7) % n)), kind == 2, kind == 0)
