"""An eager batch after a replay does not take its k1 planes from buffers that the graph has written since."""
import numpy as np
import pytest

from ephip import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,box", [(9, 5), (16, 5)])
def test_eager_batches_between_replays(backend, nw, box):
    import torch
    from ephip import eph
    m = M.make_model(nw=nw, natoms=1, box_hd=5, box_g=box, seed=50 + nw, g_dtype=np.complex64)
    st = eph.setup_outer_q(m, (20, 2, 2), (4, 2, 2), (-9.0, 9.0) if nw == 9 else (-1.2, 1.2), backend)
    plane = st.ksurv.cpu().numpy() // 4
    assert len(set(plane)) == 20

    def first(p):
        return int(np.flatnonzero(plane == p)[0])

    n = min(first(p + 2) - first(p) for p in (0, 8, 12))           # k of about two planes
    loop, fresh = eph.OuterKLoop(st, nk_batch=n), eph.OuterKLoop(st, nk_batch=n)
    assert loop.rr is not None and loop.rr.lanes()
    graph = loop.capture([first(0), first(8)], n)                  # groups 0 and 1 of eight planes
    for rep in range(3):
        for early, late in ((8, 12), (0, 4), (16, 18)):            # two batches of one group around a replay
            loop.run_kbatch(first(early), n)
            graph.replay()
            got, ref = loop.run_kbatch(first(late), n), fresh.run_kbatch(first(late), n)
            fresh.rr.invalidate()
            assert torch.equal(got.count, ref.count)
            for u, c in enumerate(ref.count.tolist()):
                a, b = got.g2[u, :c], ref.g2[u, :c]
                ok = (st.ph.omega[ref.col_index[u, :c].long()] > 1e-4).repeat(1, st.nbw)   # not the acoustic zeros
                assert bool(ok.any()) and float((a - b)[ok].abs().max()) <= 1e-6 * float(b[ok].max()), (rep, early, u)
