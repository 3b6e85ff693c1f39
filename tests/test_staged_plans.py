"""Which lists of R, k and q the staged forms take, and what they plan for them; no GPU."""
import types

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ephip import eph  # noqa: E402


def _box(n, lo=None):
    """All R of a box of edges n from lo (centred if None), R1 fastest."""
    lo = [-(m // 2) for m in n] if lo is None else lo
    r3, r2, r1 = np.meshgrid(*(np.arange(n[a]) + lo[a] for a in (2, 1, 0)), indexing="ij")
    return np.stack([r1.ravel(), r2.ravel(), r3.ravel()], axis=1).astype(np.int32)


def _grid(n):
    x = np.meshgrid(*(np.arange(m) / m for m in n), indexing="ij")
    return np.stack([v.ravel() for v in x], axis=1)


def _setup(nw=12, nm=6, kgrid=(4, 4, 6), qgrid=None, nbw=2, re=None, rp=None, seed=0):
    """The part of OuterQSetup that the plans read, every band window of nbw bands, on the CPU."""
    qgrid = kgrid if qgrid is None else qgrid
    re = _box((5, 5, 5)) if re is None else re
    rp = re if rp is None else rp
    xk, nk = torch.from_numpy(_grid(kgrid)), int(np.prod(kgrid))
    filt = types.SimpleNamespace(keep=torch.ones(nk, dtype=torch.uint8), band_min=torch.ones(nk, dtype=torch.int64),
                                 band_max=torch.full((nk,), nbw, dtype=torch.int64))
    el = types.SimpleNamespace(xk=xk, filt=filt, U=torch.zeros((nk, nw, nw), dtype=torch.complex64))
    nq = int(np.prod(qgrid))
    ph = types.SimpleNamespace(xq=torch.from_numpy(_grid(qgrid)), omega=torch.zeros((nq, nm), dtype=torch.float64),
                               u=torch.zeros((nq, nm, nm), dtype=torch.complex64))
    epmat = types.SimpleNamespace(nr=len(rp), ndata=nw * nw * nm * len(re), irvec_dev=lambda: torch.from_numpy(rp))
    return types.SimpleNamespace(el=el, ph=ph, ksurv=torch.arange(nk), nbw=nbw, epmat=epmat, nw=nw, nm=nm,
                                 irvec_el_dev=torch.from_numpy(re), kgrid=tuple(kgrid), qgrid=tuple(qgrid))


def _kr(st, **kw):
    return eph._GridOptKR.build(st, st.ksurv.numpy(), st.nw * st.nw * st.nm * st.epmat.nr, **kw)


@pytest.fixture(autouse=True)
def _no_kernels(monkeypatch):
    """The plans' phase tables are not formed here."""
    monkeypatch.setattr(eph.L, "call", lambda *a: None)
    monkeypatch.setattr(eph.L, "ptr", lambda t: None if t is None else t.data_ptr())
    monkeypatch.setattr(eph.L, "stream_handle", lambda: None)


@pytest.mark.parametrize("nw,general", [(12, True), (16, False), (8, False)])
def test_repeated_R_takes_the_direct_sums(nw, general):
    """The staged forms hold one column per R of a box: a list that names an R twice sums both."""
    r = _box((5, 5, 5))
    twice = np.ascontiguousarray(np.sort(np.concatenate([r, r[17:18]]).view("i4,i4,i4"), axis=0).view(np.int32))
    assert _kr(_setup(nw, re=r), general=general) is not None
    assert _kr(_setup(nw, re=twice), general=general) is None
    assert eph._GridOptKQ.build(_setup(nw, re=r), general=general) is not None
    assert eph._GridOptKQ.build(_setup(nw, re=r, rp=twice), general=general) is None
