"""The staged outer-q loop with a tile of q in parts (its buffers bounded) gives the bits of the whole tile."""
import numpy as np
import pytest

from ephip import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,atoms,box,kgrid,nk_batch,tile", [
    (4, 2, 5, (11, 3, 4), 50, 7),      # two groups of planes, several k batches
    (16, 1, 3, (4, 4, 4), 8192, 16),
    (7, 1, 7, (3, 5, 4), 13, 5)])      # odd rows: a part's rows start off 16 bytes
@pytest.mark.parametrize("nt", [1, 3])
def test_parts_of_a_tile(backend, monkeypatch, nw, atoms, box, kgrid, nk_batch, tile, nt):
    import torch
    from ephip import eph
    m = M.make_model(nw=nw, natoms=atoms, box_hd=5, box_g=box, seed=300 + nw, g_dtype=np.complex64)
    st = eph.setup_outer_q(m, kgrid, kgrid, (-1.5, 1.5), backend)

    class Keep(eph.AbstractCalculator):
        def __init__(self):
            self.got = []

        def run(self, p):
            self.got.append((p.iq, p.ik.clone(), p.ikq.clone(), p.g2.clone(), p.ep.clone()))

    whole = eph.OuterQLoop(st, nk_batch=nk_batch, nq_tile=tile, keep_ep=True)
    assert whole.staged.nt == tile
    one = sum(x.numel() * x.element_size() for x in (whole.staged.g2, whole.staged.ep, whole.staged.ikq, whole.staged.A))
    one = one // tile + 8 * whole.staged.go.plane_buffers() * whole.staged.go.np ** 2 * nw * nw * st.nm
    monkeypatch.setattr(eph._StagedRQ, "TILE_BYTES", nt * one)
    parts = eph.OuterQLoop(st, nk_batch=nk_batch, nq_tile=tile, keep_ep=True)
    assert parts.staged.nt == nt
    a, b = Keep(), Keep()
    for iq0, n in ((0, tile), (5, 2), (2, tile)):
        whole.run_qtile(iq0, n, [a])
        parts.run_qtile(iq0, n, [b])
    assert len(a.got) == len(b.got) > 0
    for x, y in zip(a.got, b.got):
        assert x[0] == y[0] and all(torch.equal(u.view(torch.uint8), v.view(torch.uint8)) for u, v in zip(x[1:3], y[1:3]))
        for u, v in zip(x[3:], y[3:]):   # bits, the acoustic 0 / 0 among them
            assert torch.equal(u.contiguous().view(torch.int32), v.contiguous().view(torch.int32))
