"""qs_rot_angle / qs_rot_backward on narrow registers in large batches, whose partial sums
span samples (shared angle) or are a few lanes of a block (per sample), against float64; the
bars are those of test_gpu_rot."""
import pytest
import torch

from qandle_amd._engine import plain
from tests.test_gpu_rot import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B", [(1, 2047), (1, 2 ** 16 + 3), (2, 1025), (3, 513), (4, 257), (5, 70), (7, 33), (8, 17),
                                 (9, 9), (10, 5), (11, 3)])
def test_narrow_large_batches(device, n, B):
    for bit in sorted({0, n // 2, n - 1}):
        for kind in range(3):
            _check(device, n, B, bit, kind, 0, kind != 1, False)
            _check(device, n, B, bit, kind, 0, kind == 1, kind == 2)
            if n > 1:
                _check(device, n, B, bit, kind, 1 << ((bit + 1) % n), kind != 2, kind == 0)


def test_more_samples_than_a_launch_has_blocks(device):
    """2^25 + 4099 one-qubit samples: no launch has a block of 256 threads for each, and the shared
    angle's partials (more than 2^14) are added up in two launches."""
    n, B = 1, 2 ** 25 + 4099
    gen = torch.Generator(device=device).manual_seed(0)
    g = torch.randn(B, 2, dtype=torch.complex64, device=device, generator=gen)
    st = torch.randn(B, 2, dtype=torch.complex64, device=device, generator=gen).requires_grad_(True)
    phi = torch.rand(B, device=device, generator=gen).requires_grad_(True)
    one = torch.tensor(0.4, device=device, requires_grad=True)
    for p in (phi, one):
        st.grad = None
        out = plain.RotFn.apply(st, p, n, 0, 1)
        out.backward(g)
        h = p.detach().double() / 2
        c, s = torch.cos(h), torch.sin(h)
        y, v = out.detach(), g.to(torch.complex128)
        want = torch.stack((c * v[:, 0] + s * v[:, 1], c * v[:, 1] - s * v[:, 0]), 1)
        assert ((st.grad - want).abs().amax() <= 8 * 2.0 ** -24 * want.abs().amax()).item()
        terms = torch.stack((v[:, 0].conj() * -1j * y[:, 1], v[:, 1].conj() * 1j * y[:, 0]), 1)
        ref, mag = 0.5 * terms.imag.sum(1), 0.5 * terms.abs().sum(1)
        if p.dim() == 0:
            ref, mag = ref.sum(), mag.sum()
        assert ((p.grad - ref).abs() <= 2.0 ** -20 * mag).all().item()
