"""FP32 Fourier transform: every wave tile and its edges, column lists and ragged units, against float64 sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows around 16, 32, 48, 64 and 96, columns around 64 and 128 and R around 8; the second line is large enough for the
# 32 x 128, 48 x 128, 96 x 64 and 64 x 64 tiles; boxes of more than 24 axis points go without the table
@pytest.mark.parametrize("nd,box,nunits,nk", [
    (1, 1, 1, 1), (15, 2, 3, 63), (17, 2, 2, 65), (49, 3, 1, 64), (97, 2, 1, 129), (16, 9, 1, 40),
    (31, 2, 70, 500), (47, 3, 64, 520), (190, 2, 40, 250), (64, 3, 40, 250), (108, 2, 30, 200)])
def test_fourier_c32_tiles(backend, nd, box, nunits, nk):
    import torch
    from ephip import _lib as L
    rng = np.random.default_rng(nd + nunits)
    dev = backend.torch_device
    g = np.arange(box) - box // 2
    irvec = np.array([(a, b, c) for a in g for b in g for c in g], dtype=np.int32)
    nr = len(irvec)
    op = (rng.standard_normal((nunits, nr, nd)) + 1j * rng.standard_normal((nunits, nr, nd))).astype(np.complex64)
    npt = nk + 7
    xk = rng.uniform(-1.5, 1.5, (npt, 3))
    ncol = rng.integers(0, nk + 1, nunits).astype(np.int32)
    ncol[0], ncol[-1] = nk, max(nk - 1, 1)
    cols = np.stack([np.sort(rng.permutation(npt)[:nk]) for _ in range(nunits)]).astype(np.int32)
    t = {k: torch.from_numpy(v).to(dev) for k, v in dict(op=op, ir=irvec, xk=xk, ncol=ncol, cols=cols).items()}
    out = torch.full((nunits, nk, nd), 7.0, dtype=torch.complex64, device=dev)
    L.call("ephip_fourier_batched_c32", nd, nr, L.ptr(t["op"]), nd, nd * nr, L.ptr(t["ir"]), L.ptr(t["xk"]), nunits, nk,
           L.ptr(t["ncol"]), L.ptr(t["cols"]), nk, L.ptr(out), nd, nk * nd, L.PREC_FP32, L.stream_handle())
    got = out.cpu().numpy()
    for u in {0, nunits // 2, nunits - 1}:
        ph = np.exp(2j * np.pi * (xk[cols[u, :ncol[u]]] @ irvec.T))
        ref = ph @ op[u].astype(np.complex128)
        # phases: three FP32 factors and two products, 1.5e-6; the sum: 2 nr roundings of 6e-8
        tol = np.abs(op[u]).sum(0).max() * (1.5e-6 + 2 * nr * 6e-8)
        assert np.abs(got[u, :ncol[u]] - ref).max(initial=0) < tol
        assert np.all(got[u, ncol[u]:] == 7.0)
