"""FP64 Fourier transform: every wave tile and its edges against the sum in long double and the tile-free variant."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows, R and columns around 8, 16 and 32 x waves, 8, 16 and 32 R a stage, and 16, 32 and 64 columns; the last six
# are large enough for the 32 x 32 tiles, one and two column waves, and the 16 x 16 ones
@pytest.mark.parametrize("nd,nr,nk", [(1, 1, 1), (8, 32, 16), (9, 33, 17), (31, 7, 15), (33, 65, 31), (64, 31, 40),
                                      (49, 64, 16500), (65, 8, 16000), (192, 9, 6176), (257, 17, 4001), (192, 40, 4100),
                                      (143, 41, 13820), (17, 65, 13801)])
def test_fourier_c64_tiles(backend, nd, nr, nk):
    import torch
    from ephip import core, tune
    rng = np.random.default_rng(nd + nr)
    dev = backend.torch_device
    irvec = rng.integers(-5, 6, (nr, 3)).astype(np.int32)
    op = rng.standard_normal((nr, nd)) + 1j * rng.standard_normal((nr, nd))
    xk = rng.uniform(-1.5, 1.5, (nk, 3))
    w = core.WannierObject(irvec, op, ndata=nd, check=False).to_device(backend, torch.complex128)
    x = torch.from_numpy(xk).to(dev)
    out = torch.full((nk + 1, nd), 7.0, dtype=torch.complex128, device=dev)
    core.fourier_batched(w, x, out=out[:nk])
    assert bool((out[nk] == 7.0).all())
    try:
        tune.set_variant(2, 1)          # 64 rows x 64 columns a workgroup, every wave in one role
        ref = core.fourier_batched(w, x)
    finally:
        tune.set_variant(2, 0)
    assert torch.equal(out[:nk], ref)   # the same sums in the same order
    cols = np.unique(rng.integers(0, nk, 24))
    arg = (irvec.astype(np.longdouble) @ xk[cols].T.astype(np.longdouble)) * 2
    ph = np.cos(np.pi * arg.astype(np.longdouble)) + 1j * np.sin(np.pi * arg.astype(np.longdouble))
    exact = op.T.astype(np.clongdouble) @ ph.astype(np.clongdouble)
    got = out[:nk].cpu().numpy()[cols].T
    # each of nr products of size <= |op|: argument rounded at |R.x| <= 22.5, then 2 nr roundings of the sum
    tol = np.abs(op).sum(0).max() * 2.3e-16 * (2 * np.pi * 22.5 * 3 + 2 * nr)
    assert np.abs(got - exact.astype(np.complex128)).max() < tol
