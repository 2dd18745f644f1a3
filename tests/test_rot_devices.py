"""A rotation whose angle is on another device than its state is refused before the kernel, which
would read the angle's address, is launched."""
import types

import pytest
import torch

from qandle_amd._engine import plain
from qandle_amd._engine.lib import EngineError


@pytest.mark.parametrize("shape", [(), (2,)])
def test_angle_on_another_device(shape, monkeypatch):
    launched = []
    monkeypatch.setattr(plain.L, "load", lambda: types.SimpleNamespace(qs_rot_angle=lambda *a: launched.append(a) or 0))
    monkeypatch.setattr(plain.L, "stream_of", lambda t: 0)
    state = torch.zeros(2, 4, dtype=torch.complex64)
    phi = torch.empty(shape, device="meta")
    with pytest.raises(EngineError):
        plain.RotFn.apply(state, phi, 2, 0, 0)
    with pytest.raises(EngineError):
        plain.ControlledRotFn.apply(state, phi, 2, 0, 0, 2)
    assert not launched
    plain.RotFn.apply(state, torch.zeros(shape), 2, 0, 0)
    assert len(launched) == 1
