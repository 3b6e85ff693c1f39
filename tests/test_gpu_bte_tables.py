"""ephip_bte_accumulate_tables against the per-term ephip_bte_accumulate_units on the same synthetic payload."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("smearing,nT,nm,nbw,one_width", [(1, 1, 12, 2, True), (1, 3, 3, 1, True), (2, 2, 5, 3, True),
                                                          (1, 4, 6, 5, False), (2, 7, 8, 2, False)])
def test_tables_match_per_term(backend, method, smearing, nT, nm, nbw, one_width):
    import torch
    from ephip import _lib as L
    rng = np.random.default_rng(17 * method + nT)
    dev = backend.torch_device
    nk, nq, nu, cs = 300, 700, 5, 700
    nb = rng.integers(0, nbw + 1, nk)
    bmin = np.where(nb > 0, rng.integers(1, 4, nk), 0)
    bmax = np.where(nb > 0, bmin + nb - 1, 0)
    off = np.concatenate([[0], np.cumsum(nb)])
    n = int(off[-1])
    es = rng.uniform(-0.3, 0.3, n)
    omega = rng.uniform(0.0, 0.1, (nq, nm))
    omega[rng.random((nq, nm)) < 0.1] = 0.0                # below the cutoff (the boson factor diverges there)
    count = np.array([700, 0, 1, 256, 257])
    col = np.stack([np.sort(rng.permutation(nq)) for _ in range(nu)])
    ikq = rng.choice(np.flatnonzero(nb > 0), (nu, cs))
    ikq[0, 5] = np.flatnonzero(nb == 0)[0]                 # a final k without a window band
    g2 = rng.uniform(0, 1, (nu, cs, nbw, nm))
    usi = rng.integers(0, n, nu)
    rowptr = np.concatenate([[0], np.cumsum(count)])
    Ts = np.linspace(0.01, 0.06, nT)
    mus = rng.uniform(-0.02, 0.02, nT)
    etas = np.full(nT, 0.03) if one_width else rng.uniform(0.005, 0.05, nT)

    def t(x, d):
        return torch.from_numpy(np.ascontiguousarray(x)).to(dev, dtype=d)

    i64, i32, f64 = torch.int64, torch.int32, torch.float64
    dcount, dcol, dikq, dg2 = t(count, i32), t(col, i32), t(ikq, i32), t(g2, torch.float32)
    dusi, doff, dbmin, dbmax = t(usi, i64), t(off, i64), t(bmin, i64), t(bmax, i64)
    des, dom, dmu, dT, deta, drow = t(es, f64), t(omega, f64), t(mus, f64), t(Ts, f64), t(etas, f64), t(rowptr, i64)
    out = []
    tab_q = torch.empty((1 + nT) * nm * nq, dtype=f64, device=dev)
    tab_s = torch.empty(nT * n, dtype=f64, device=dev)
    for tables in (False, True):
        S_out = torch.zeros((nT, n), dtype=f64, device=dev)
        S_in = torch.full((int(rowptr[-1]), nbw, nT), 9.0, dtype=f64, device=dev)
        code = torch.zeros(int(rowptr[-1]), dtype=i32, device=dev)
        head = [L.ptr(dcount), L.ptr(dcol), L.ptr(dikq), L.ptr(dg2), L.ptr(dusi), L.ptr(doff), L.ptr(dbmin), L.ptr(dbmax)]
        tail = [method, smearing, 1e-5, n, L.ptr(drow), L.ptr(S_out), L.ptr(S_in), L.ptr(code), L.stream_handle()]
        if tables:
            L.call("ephip_bte_tables", nq, nm, L.ptr(dom), n, L.ptr(des), nT, L.ptr(dmu), L.ptr(dT), method, L.ptr(tab_q),
                   L.ptr(tab_s), L.stream_handle())
            L.call("ephip_bte_accumulate_tables", nu, cs, nbw, nm, nq, *head, L.ptr(des), L.ptr(tab_q), L.ptr(tab_s),
                   1.0 / nq, nT, L.ptr(dT), L.ptr(deta), *tail)
        else:
            L.call("ephip_bte_accumulate_units", nu, cs, nbw, nm, *head, L.ptr(des), L.ptr(dom), 1.0 / nq, nT, L.ptr(dmu),
                   L.ptr(dT), L.ptr(deta), *tail)
        out.append((S_out.cpu().numpy(), S_in.cpu().numpy(), code.cpu().numpy()))
    (so, si, c), (so2, si2, c2) = out
    assert np.array_equal(c, c2)
    # terms of one sign or another (methods 1 and 6 subtract): 1e-11 of the largest value
    for a, b in ((so, so2), (si, si2)):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 1e-11 * np.abs(a).max()
