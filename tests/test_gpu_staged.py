"""The staged outer-k transforms for any model shape (csrc/staged.hip) against the direct Fourier kernels: kept lists
exact, g2 to 1e-5 of its largest value (both sum in FP32; each is within 1e-6 of the 64-bit result)."""
import dataclasses

import numpy as np
import pytest

from ephip import model as M

pytestmark = pytest.mark.gpu


def _cut(m, axis_min):
    """The model without the R below axis_min on each axis (an uneven box; None leaves an axis alone)."""
    keep = np.all([np.ones(len(m.irvec_el), bool) if lo is None else m.irvec_el[:, a] >= lo
                   for a, lo in enumerate(axis_min)], axis=0)
    n = len(m.irvec_el)
    ep = m.epmat_ph.reshape(n, n, -1)[keep][:, keep]
    r = np.ascontiguousarray(m.irvec_el[keep])
    return dataclasses.replace(m, irvec_el=r, irvec_ep=r.copy(), epmat_ph=np.ascontiguousarray(ep.reshape(len(r), -1)))


# nw, atoms, g box, first R kept per axis, k grid, q grid, window
CASES = [
    (1, 1, 5, None, (6, 5, 4), (6, 5, 4), 4.0),            # one orbital: three idle j, one row per mode
    (3, 1, 5, None, (5, 7, 3), (5, 7, 3), 1.5),
    (4, 1, 7, None, (6, 6, 6), (3, 6, 2), 1.0),            # one wave, q grid a divisor of the k grid
    (5, 2, 5, (None, -1, None), (4, 4, 6), (4, 4, 6), 1.2),  # face 5 x 4, not symmetric, index map
    (6, 1, 5, (-1, -1, -1), (4, 4, 4), (4, 4, 4), 1.2),    # 4^3 box: dense and not symmetric
    (7, 2, 7, (None, None, -2), (4, 5, 4), (4, 5, 4), 1.0),  # face 7 x 6
    (8, 2, 5, None, (8, 8, 8), (8, 8, 8), 1.0),
    (12, 3, 5, None, (6, 5, 4), (6, 5, 4), 0.6),
    (13, 1, 5, None, (4, 4, 4), (4, 4, 4), 3.0),           # wide: four and more bands a thread
    (16, 4, 5, None, (4, 6, 4), (4, 6, 4), 2.5),
    (16, 6, 5, None, (4, 4, 4), (4, 4, 4), 0.6),           # 18 modes
    (20, 1, 5, None, (4, 4, 4), (2, 4, 4), 1.0),
    (32, 1, 5, None, (4, 4, 2), (4, 4, 2), 1.5),
    (4, 1, 5, None, (1, 24, 24), (1, 24, 24), 6.0),        # 576 kept q per slab: several segments, cut lines
    (9, 1, 5, None, (2, 3, 64), (2, 3, 64), 2.0),          # lines of 64 q; line pieces on the k side
]


@pytest.mark.parametrize("nw,atoms,box,cut,kgrid,qgrid,window", CASES)
def test_staged_against_direct(backend, nw, atoms, box, cut, kgrid, qgrid, window):
    import torch
    from ephip import _lib as L
    from ephip import eph
    m = M.make_model(nw=nw, natoms=atoms, box_hd=5, box_g=box, seed=900 + nw, g_dtype=np.complex64)
    if cut is not None:
        m = _cut(m, cut)
    st = eph.setup_outer_q(m, kgrid, qgrid, (-window, window), backend)
    nks = st.ksurv.shape[0]
    assert nks > 0
    nb = max(1, (nks + 1) // 2)
    staged = eph.OuterKLoop(st, nk_batch=nb, precision=L.PREC_FP32, with_ep=True)
    direct = eph.OuterKLoop(st, nk_batch=nb, precision=L.PREC_FP32, gridopt=False)
    assert staged.rr.general or nw == 16
    assert staged.kq.general or (nw == 16 and st.nbw <= 4 and m.nmodes <= 16)
    for i0 in (0, nks - nb, nb % nks, 0):    # advancing and returning batches
        for t in (staged.g2, direct.g2):
            t.fill_(7.0)
        ps, pd = staged.run_kbatch(i0, nb), direct.run_kbatch(i0, nb)
        assert torch.equal(ps.count, pd.count) and torch.equal(ps.unit_state, pd.unit_state)
        cnt = ps.count.cpu().numpy()
        num = den = 0.0
        for u in range(len(cnt)):
            c = cnt[u]
            assert torch.equal(ps.col_index[u, :c], pd.col_index[u, :c]) and torch.equal(ps.ikq[u, :c], pd.ikq[u, :c])
            a, b = ps.g2[u, :c].double(), pd.g2[u, :c].double()
            ok = (st.ph.omega[ps.col_index[u, :c].long()] > 1e-4).repeat(1, st.nbw)   # not the acoustic zeros
            num = max(num, float(((a - b).abs() * ok).max()) if c else 0.0)
            den = max(den, float((b * ok).max()) if c else 0.0)
            assert torch.equal(a == 0, b == 0)                                       # zeros past the k+q window
            w = 2 * st.ph.omega[ps.col_index[u, :c].long()].repeat(1, st.nbw)
            e2 = ps.ep[u, :c].abs().double().square()
            assert bool(((e2 / w - a).abs() <= 1e-5 * (a.abs() + 1e-30))[ok].all())
        assert den > 0 and num <= 1e-5 * den, num / den


def test_staged_entries_refuse_what_they_do_not_cover(backend):
    import ctypes as C
    from ephip import _lib as L
    q = (C.c_int32 * 3)(4, 4, 4)
    big = (C.c_int32 * 3)(4, 65, 4)

    def kq(nw=4, nm=3, nbw=2, n1=5, np_=5, grid=q, nunits=1):
        L.call("ephip_staged_kq", nw, nm, nbw, nunits, n1, np_, -2, -2, -2, None, C.addressof(grid), None, None, None,
               None, nw * nm * 125, nw * nm, None, None, None, 64, None, None, None, None, None, None, 8.0, 1.0, None,
               None, None)

    for kw, msg in [(dict(nw=33), "nw=33"), (dict(nm=49), "nm=49"), (dict(nbw=5), "nbw=5"), (dict(np_=9), "Rp box"),
                    (dict(n1=33), "Rp box"), (dict(grid=big), "q grid"), (dict(), "null device pointer")]:
        with pytest.raises(L.EphipError, match=msg):
            kq(**kw)
    kq(nunits=0)


@pytest.mark.parametrize("nw,atoms,box,cut,kgrid,qgrid,window,tile,nk_batch", [
    (1, 1, 3, None, (4, 5, 4), (4, 5, 4), 4.0, 3, 8),
    (3, 1, 5, None, (5, 7, 3), (5, 7, 3), 1.5, 17, 1000),       # odd rows: no paired loads; two launches of q columns
    (4, 1, 7, (None, -2, -1), (4, 6, 4), (2, 6, 4), 1.0, 16, 13),  # uneven box, several k batches
    (7, 2, 5, None, (4, 4, 4), (4, 4, 4), 1.5, 5, 40),
    (16, 4, 3, None, (4, 4, 4), (2, 2, 2), 1.5, 8, 8192),
    (13, 6, 5, None, (4, 3, 4), (4, 3, 4), 2.5, 4, 20),          # 18 modes, wide window
    (32, 1, 3, None, (3, 4, 2), (3, 4, 2), 1.0, 2, 5),
])
def test_staged_outer_q_against_direct(backend, nw, atoms, box, cut, kgrid, qgrid, window, tile, nk_batch):
    import torch
    from ephip import eph
    m = M.make_model(nw=nw, natoms=atoms, box_hd=5, box_g=box, seed=700 + nw, g_dtype=np.complex64)
    if cut is not None:
        m = _cut(m, cut)
    st = eph.setup_outer_q(m, kgrid, qgrid, (-window, window), backend)
    nq = st.ph.xq.shape[0]
    staged = eph.OuterQLoop(st, nk_batch=nk_batch, nq_tile=tile, keep_ep=True)
    direct = eph.OuterQLoop(st, nk_batch=nk_batch, nq_tile=tile, keep_ep=True, staged=False)
    assert staged.staged is not None and direct.staged is None

    class Keep(eph.AbstractCalculator):
        def __init__(self):
            self.got = []

        def run(self, p):
            self.got.append((p.iq, p.ik.clone(), p.ikq.clone(), p.g2.clone(), p.ep.clone()))

    a, b = Keep(), Keep()
    for iq0, n in ((0, min(tile, nq)), (nq - 1, 1), (1, min(tile, nq - 1))):   # whole, single and partial tiles
        staged.run_qtile(iq0, n, [a])
        direct.run_qtile(iq0, n, [b])
    assert len(a.got) == len(b.got)
    num = den = 0.0
    for x, y in zip(a.got, b.got):
        assert x[0] == y[0] and torch.equal(x[1], y[1]) and torch.equal(x[2], y[2])
        ok = st.ph.omega[x[0]] > 1e-4
        assert torch.equal(x[3] == 0, y[3] == 0)
        if not bool(ok.any()):   # q = 0 of one atom: acoustic modes only
            continue
        g, r = x[3].double()[:, ok], y[3].double()[:, ok]
        num, den = max(num, float((g - r).abs().max())), max(den, float(r.max()))
        e2 = x[4].abs().double().square()[:, ok] / (2 * st.ph.omega[x[0]][ok]).view(1, -1, 1, 1)
        assert bool(((e2 - g).abs() <= 1e-5 * (g.abs() + 1e-30)).all())
    assert den > 0 and num <= 1e-5 * den, num / den
