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


@pytest.mark.parametrize("offset,fused", [(0, True), (1, False), (2, False), (4, True)])
def test_parameters_off_16_bytes_take_the_layers(calls, offset, fused):
    """The fused step reads the parameters four at a time; a view into another vector may start anywhere."""
    net = surrogate.BandSurrogate(3, torch.device("cpu"))
    own = torch.from_numpy(np.zeros(net.nparam + 8, np.float32))
    base = (-own.data_ptr() // 4) % 4
    net.p = own[base + offset: base + offset + net.nparam]
    net.loss_and_grad(torch.zeros((5, 3), dtype=torch.float64), torch.zeros((5, 16)))
    assert ("ephip_mlp_train_step" in calls) == fused and calls


def test_buffers_of_the_other_form_are_completed(calls):
    """The two forms need other workspaces; buffers returned by one serve the other."""
    net = surrogate.BandSurrogate(3, torch.device("cpu"))
    xk, t = torch.zeros((2000, 3), dtype=torch.float64), torch.zeros((2000, 16))
    own = torch.zeros(net.nparam + 8)
    views = [own[o: o + net.nparam] for o in range(2)]
    for first in views:
        net.p = first
        _, acts, grads = net.loss_and_grad(xk, t)
        net.p = next(v for v in views if v is not first)
        _, _, got = net.loss_and_grad(xk, t, acts, grads)
        need = 63 * net.nparam if net._fused() else 64 * 128 * 128   # 63 workgroups of at least 32 points
        assert got["part"].numel() >= need and got["gy"] is grads["gy"]
        assert net._fused() or got["ones"].numel() == 2000
