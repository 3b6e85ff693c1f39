"""The fused vector work of an iteration of the BTE solve (csrc/bte.hip) against the same in extended precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one block and its remainder, the last grid without a stride loop and the first with one
@pytest.mark.parametrize("n", [0, 1, 255, 257, 65536, 65537, 200003])
@pytest.mark.parametrize("update", [False, True])
def test_bte_step(backend, n, update):
    import torch
    from ephip import _lib as L
    rng = np.random.default_rng(n + update)
    dev = backend.torch_device
    y, rhs, df, vs = (rng.standard_normal((n, 3)) for _ in range(4))
    inv_tau = rng.uniform(0.5, 2.0, n)
    old = rng.standard_normal(10)
    d = {k: torch.from_numpy(v.copy()).to(dev) for k, v in dict(y=y, rhs=rhs, df=df, vs=vs, it=inv_tau, old=old).items()}
    buf = torch.full((9 * 256 + 11,), 7.0, dtype=torch.float64, device=dev)
    out = buf[9 * 256:]
    mix, scale = 0.7, 0.37
    L.call("ephip_bte_step", n, L.ptr(d["y"]) if update else None, L.ptr(d["it"]), L.ptr(d["rhs"]), mix, L.ptr(d["df"]),
           L.ptr(d["vs"]), scale, L.ptr(d["old"]), L.ptr(buf), L.ptr(out), L.stream_handle())
    ld = np.longdouble
    ref = df.astype(ld)
    if update:
        ref = (y.astype(ld) / inv_tau[:, None] + rhs) * ld(mix) + ref * (1 - ld(mix))
    got = d["df"].cpu().numpy()
    eps = 2.3e-16
    assert np.abs(got - ref).max(initial=0) <= 6 * eps * (np.abs(y).max(initial=0) * 2 + np.abs(rhs).max(initial=0)
                                                          + np.abs(df).max(initial=0))
    o = out.cpu().numpy()
    assert o[10] == 7.0
    exact = scale * (got.astype(ld).T @ vs.astype(ld))
    # sums of n / 65536 + 1 terms a thread, then of at most 64 x 4 x 256 by trees
    tol = eps * scale * (np.abs(got).T @ np.abs(vs)).max(initial=0) * (n / 65536 + 24)
    assert np.abs(o[:9].reshape(3, 3) - exact).max() <= tol
    if n:
        diff = np.linalg.norm(o[:9] - old[:9]) / np.linalg.norm(o[:9])
        assert abs(o[9] - diff) <= 30 * eps * diff
