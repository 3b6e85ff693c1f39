"""Stage 1 of the staged RR->kR in groups of fewer planes (where memory is short) against the usual groups."""
import numpy as np
import pytest

from ephip import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,box", [(16, 7), (6, 5), (8, 5)])
@pytest.mark.parametrize("planes", [1, 3])
def test_groups_of_fewer_planes(backend, nw, box, planes):
    import torch
    from ephip import eph
    m = M.make_model(nw=nw, natoms=1, box_hd=5, box_g=box, seed=40 + nw, g_dtype=np.complex64)
    st = eph.setup_outer_q(m, (11, 4, 3), (11, 4, 3), (-1.0, 1.0), backend)
    nks = st.ksurv.shape[0]
    usual, few = (eph.OuterKLoop(st, nk_batch=20) for _ in range(2))
    few.rr.PLANES = planes
    for i0 in (*range(0, nks, 20), 0, 40):
        for t in (usual.g2, few.g2):
            t.fill_(7.0)
        a, b = usual.run_kbatch(i0, 20), few.run_kbatch(i0, 20)
        ok = torch.isfinite(a.g2)
        assert torch.equal(ok, torch.isfinite(b.g2))
        # each plane's sums run in the same order; 1e-5 as between the staged and the direct form
        assert float((a.g2 - b.g2)[ok].abs().max()) <= 1e-5 * float(a.g2[ok].max())
