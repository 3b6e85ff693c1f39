"""Which gradients of the band-energy network take the fused step; no GPU."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ephip import surrogate  # noqa: E402


@pytest.fixture
def calls(monkeypatch):
    names = []
    monkeypatch.setattr(surrogate.L, "call", lambda name, *a: names.append(name))
    monkeypatch.setattr(surrogate.L, "ptr", lambda t: None if t is None else t.data_ptr())
    monkeypatch.setattr(surrogate.L, "stream_handle", lambda: None)
    return names


def test_no_points_are_refused(calls):
    """No point has no mean error, and the gradient of an earlier call would stay in place."""
    net = surrogate.BandSurrogate(3, torch.device("cpu"))
    with pytest.raises((ZeroDivisionError, surrogate.L.EphipError)):
        net.loss_and_grad(torch.zeros((0, 3), dtype=torch.float64), torch.zeros((0, 16)))
