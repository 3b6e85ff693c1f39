"""The fused gradient (csrc/mlp_train.hip) against the layer-by-layer kernels of the same network."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,nf2,hidden,n", [(16, 32, 128, 1000), (3, 8, 16, 1), (20, 16, 32, 17), (40, 64, 96, 333),
                                             (64, 24, 112, 2049), (16, 64, 128, 5000), (5, 16, 64, 144)])
def test_train_step_matches_layers(backend, nw, nf2, hidden, n):
    import torch
    from ephip.surrogate import BandSurrogate
    rng = np.random.default_rng(nw + n)
    dev = backend.torch_device
    xk = torch.from_numpy(rng.uniform(-0.5, 1.5, (n, 3))).to(dev)
    E = torch.from_numpy(np.sort(rng.standard_normal((n, nw)), axis=1)).to(dev)
    net = BandSurrogate(nw, dev, nf2=nf2, hidden=hidden, seed=n)
    for b in ("b1", "b2", "b3"):
        v = net.view(net.p, b)
        v.copy_(torch.from_numpy(rng.standard_normal(v.numel()).astype(np.float32)).to(dev))
    t = net.targets(E)
    assert net._fused()
    loss, acts, gw = net.loss_and_grad(xk, t)
    g = net.g.clone()
    loss2, _, _ = net.loss_and_grad(xk, t, acts, gw)      # into the same buffers
    assert torch.equal(loss, loss2) and torch.equal(net.g, g)
    net._fused = lambda: False
    rloss, racts, rgw = net.loss_and_grad(xk, t)
    for k in racts:                                       # the same sums in the same order
        assert torch.equal(acts[k], racts[k]), k
    assert torch.equal(gw["gy"], rgw["gy"])
    assert float((loss - rloss).abs().max()) <= 1e-14 * float(rloss.max())
    # FP32 sums of n products in two orders: a few ulp of the gradient's scale times sqrt(n)
    assert float((g - net.g).norm()) <= 1e-5 * float(net.g.norm())


def test_train_step_refuses_other_sizes(backend):
    import torch
    from ephip import _lib as L
    from ephip.surrogate import BandSurrogate
    dev = backend.torch_device
    for kw in (dict(nf2=32, hidden=136), dict(nf2=30, hidden=64), dict(nf2=72, hidden=64)):
        assert not BandSurrogate(4, dev, **kw)._fused()
    x = torch.zeros(64, device=dev)
    with pytest.raises(L.EphipError, match="multiples of 16"):
        L.call("ephip_mlp_train_step", 4, L.ptr(x), 32, L.ptr(x), 136, 16, *([L.ptr(x)] * 12), 1, L.ptr(x), L.ptr(x),
               L.stream_handle())
