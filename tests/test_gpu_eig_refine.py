"""Several matrices a wave in the FP64 refinement: one, two or four by n and the batch."""
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
