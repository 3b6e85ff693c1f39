"""Several matrices a wave in the FP32 eigensolve (by n) and the FP64 refinement (by n and the batch)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(n, nb, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((nb, n, n)) + 1j * rng.standard_normal((nb, n, n))
    h = a + np.conj(np.transpose(a, (0, 2, 1)))
    if n >= 4:
        h[::3, 1, :] = h[::3, :, 1] = 0     # a decoupled level: it stays decoupled through every rotation
        h[::3, 1, 1] = 0.5
        h[::5] = np.eye(n) * 0.25           # every eigenvalue the same
    return h


@pytest.mark.parametrize("n", [9, 12, 15, 16])
def test_refine_same_bits_for_any_batch(backend, n):
    """Batches of up to 1024 go one matrix a wave, larger ones two: the same matrix gives the same bits, also as the
    odd last one."""
    import torch
    from ephip import core
    nb = 1027
    hc = torch.from_numpy(np.ascontiguousarray(np.transpose(_batch(n, nb, n), (0, 2, 1)))).cuda()
    E, U = core.eigen_batched_refined(hc)
    Ea, Ua = core.eigen_batched_refined(hc[:1024].contiguous())
    Eb, Ub = core.eigen_batched_refined(hc[1024:].contiguous())
    assert torch.equal(E, torch.cat([Ea, Eb])) and torch.equal(U, torch.cat([Ua, Ub]))


@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 16, 17])
@pytest.mark.parametrize("nb", [1, 2, 3, 5])
def test_refine_partial_waves(backend, n, nb):
    """Waves with fewer matrices than they take: eigenvalues to a few ulp of the norm, and vectors to FP32 rounding."""
    import torch
    from ephip import core
    h = _batch(n, nb, 50 + n)
    hc = torch.from_numpy(np.ascontiguousarray(np.transpose(h, (0, 2, 1)))).cuda()
    E, U = core.eigen_batched_refined(hc)
    E, U = E.cpu().numpy(), U.cpu().numpy()
    for b in range(nb):
        w = np.linalg.eigvalsh(h[b])
        assert np.abs(E[b] - w).max() < 1e-13 * max(np.abs(w).max(), 1.0)
        V = U[b].T.astype(np.complex128)
        assert np.abs(h[b] @ V - V * E[b]).max() < 1e-6 * max(np.abs(w).max(), 1.0)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 16, 17, 32])
def test_heev_mixed_matrices_in_a_wave(backend, n):
    """Matrices that take different ways through the QL iteration side by side in a wave (dense, decoupled, diagonal,
    zero, and scaled so that squares leave the range in which hypot and the quotients need no scaling): each gives the
    bits that it gives alone."""
    import torch
    from ephip import core
    h = _batch(n, 45, 70 + n)
    h[2::9] *= 2.0 ** -70
    h[4::9] *= 2.0 ** 55
    h[6::9] = 0
    h[7::9] = np.eye(n) * np.arange(n)
    hc = torch.from_numpy(np.ascontiguousarray(np.transpose(h, (0, 2, 1)).astype(np.complex64))).cuda()
    E, U = core.eigen_batched(hc)
    assert torch.equal(E, core.eigvals_batched(hc))
    for b in range(45):
        Eb, Ub = core.eigen_batched(hc[b:b + 1].contiguous())
        assert torch.equal(Eb[0], E[b]) and torch.equal(Ub[0], U[b])
