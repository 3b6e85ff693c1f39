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


@pytest.mark.parametrize("nw,general", [(9, True), (16, False)])
@pytest.mark.parametrize("order", ["grid", "shuffled", "two_passes"])
def test_projection_covers_every_line_in_any_order_of_k(monkeypatch, nw, general, order):
    """Each line of the surviving k goes to one launch, from its own plane's sums, whatever the order of the k."""
    import ctypes as C
    st = _setup(nw, 3, (19, 2, 3))
    ks = np.arange(19 * 6)
    if order == "shuffled":
        np.random.default_rng(1).shuffle(ks)
    elif order == "two_passes":
        ks = np.concatenate([ks[::2], ks[1::2]])
    st.ksurv = torch.from_numpy(ks)
    go = _kr(st, general=general)
    assert go.lanes()
    nk, nb = len(ks), st.nbw
    k_units = torch.arange(nk + 1, dtype=torch.int32) * nb
    loop = types.SimpleNamespace(st=st, xk_surv=st.el.xk[st.ksurv], k_unit_start_dev=k_units,
                                 unit_kpos=torch.zeros(nk * nb, dtype=torch.int32),
                                 unit_state=torch.zeros(nk * nb, dtype=torch.int64),
                                 unit_band=torch.zeros(nk * nb, dtype=torch.int32), max_units=nk * nb, nk_batch=nk,
                                 epmat_el=torch.zeros((len(st.irvec_el_dev), go.nd), dtype=torch.complex64))
    holds, done = {}, []                                # plane coordinate of each buffer, lines projected

    def call(name, *a):
        if name == "ephip_gridopt_stage1_planes":
            n = a[9]
            x1 = (C.c_double * n).from_address(a[10])
            out = (C.c_void_p * n).from_address(a[12])
            holds.update({out[p]: x1[p] for p in range(n)})
        elif name == "ephip_lane_project":
            m = a[4]
            op1, la, lz = ((t * m).from_address(x) for t, x in zip((C.c_void_p, C.c_int32, C.c_int32), a[5:8]))
            assert 1 <= m <= 8
            for p in range(m):
                for line in range(la[p], lz[p]):
                    k = int(go.line_start_host[line])
                    assert holds[op1[p]] == float(loop.xk_surv[k, 0])
                    done.append(line)

    monkeypatch.setattr(eph.L, "call", call)
    go.run(loop, 0, nk, 0, nk * nb, torch.zeros((nk * nb, 1), dtype=torch.complex64), None)
    assert sorted(done) == list(range(len(go.line_start_host) - 1))


@pytest.mark.parametrize("nw,general", [(12, True), (16, False)])
def test_points_off_the_grid_take_the_direct_sums(nw, general):
    """kR->kq takes the q from their place in the grid, RR->kR a plane's and a line's coordinate from one k."""
    def plans(st):
        return _kr(st, general=general) is not None, eph._GridOptKQ.build(st, general=general) is not None

    assert plans(_setup(nw)) == (True, True)
    st = _setup(nw)
    st.ph.xq, st.el.xk = st.ph.xq - 1.0, st.el.xk + torch.tensor([0.01, 0.02, 0.03])   # whole cells; a shift of all k
    assert plans(st) == (True, True)
    st = _setup(nw)
    st.ph.xq = st.ph.xq + torch.tensor([0.0, 0.0, 0.1])
    assert plans(st) == (True, False)
    for some in (slice(0, 7), torch.randperm(96, generator=torch.Generator().manual_seed(0))):  # some q, another order
        st = _setup(nw)
        st.ph.xq = st.ph.xq[some]
        assert plans(st) == (True, False)
    for axis, ok in ((0, False), (1, False), (2, True)):   # one k off its plane, off its line, elsewhere on its line
        st = _setup(nw)
        st.el.xk[10, axis] += 0.05
        assert plans(st) == (ok, True)


@pytest.mark.parametrize("staged", [True, False])
def test_outer_q_tile_past_the_last_q_is_refused(monkeypatch, staged):
    """A tile reads its q, phonons and frequencies by position: it has to lie within the list and the buffers."""
    st = _setup(3, 3, (4, 2, 3))
    st.epmat.op_r = torch.zeros((1, 1))
    loop = eph.OuterQLoop(st, nq_tile=8, staged=staged)
    assert (loop.staged is not None) == staged
    nq, calls = st.ph.xq.shape[0], []
    monkeypatch.setattr(eph.L, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(eph, "get_eph_RR_to_Rq_batched", lambda *a, **k: calls.append("RR_to_Rq"))
    for iq0, n in ((nq - 3, 4), (nq, 1), (-1, 2), (0, 9), (0, -1)):
        with pytest.raises((eph.L.EphipError, IndexError)):
            loop.run_qtile(iq0, n)
        assert not calls


@pytest.mark.parametrize("nbw", [1, 3, 4])
@pytest.mark.parametrize("edge", [4, 5])   # a face without its opposite offsets, and one with them
def test_line_pieces_fit_the_projection(edge, nbw):
    """ephip_staged_project takes pieces of at most 64 k and 128 units: 8 orbitals, lines of 48 k."""
    st = _setup(8, 3, (2, 2, 48), (1, 1, 1), nbw=nbw, re=_box((edge,) * 3))
    st.epmat.op_r = torch.zeros((1, 1))
    rr = eph.OuterKLoop(st, nk_batch=192).rr
    assert rr.general and rr.lanes() == (edge == 5)
    assert rr.max_line_units <= 128 and rr.max_line_k <= 64
    assert rr.line_start_host[0] == 0 and rr.line_start_host[-1] == 192


def _outer_q(st, **kw):
    st.epmat.op_r = torch.zeros((1, 1))
    return eph.OuterQLoop(st, **kw)


@pytest.mark.parametrize("keep_ep", [False, True])
@pytest.mark.parametrize("tile,budget", [(8, 1 << 33), (8, 3 << 20), (8, 1 << 20), (5, 1 << 18)])
def test_outer_q_buffers_stay_within_their_budget(monkeypatch, keep_ep, tile, budget):
    """What the staged form holds for every surviving k of a tile is bounded: fewer q at a time, or the direct form,
    whose buffers are nk_batch rows."""
    monkeypatch.setattr(eph._StagedRQ, "TILE_BYTES", budget)
    st = _setup(4, 6, (6, 5, 4), nbw=3)
    loop = _outer_q(st, nq_tile=tile, nk_batch=50, keep_ep=keep_ep)
    s = loop.staged
    per_q = 120 * (6 * 9 * (12 if keep_ep else 4) + 8) + 8 * 150 * 4 * 6 + 8 * 6 * 25 * 4 * 4 * 6   # 6 planes of k1
    if per_q > budget:
        assert s is None
        return
    assert s.nt == min(tile, budget // per_q)
    held = [s.g2, s.ikq, s.A] + ([s.ep] if keep_ep else [])
    held = sum(t.numel() * t.element_size() for t in held) + 8 * 6 * 25 * s.go.nd_max
    assert held <= budget and s.go.nd_max == s.nt * 4 * 4 * 6


@pytest.mark.parametrize("quarter,planes", [(100, 8), (13, 6), (2, 1), (1, 0)])
def test_outer_k_planes_leave_room(monkeypatch, quarter, planes):
    """Plane buffers take at most a quarter of what the "el" tensor leaves: smaller groups, or the direct form; the
    batch is planned on what they leave."""
    st = _setup(9, 3, (19, 2, 3))
    st.epmat.op_r = torch.zeros((125, st.epmat.ndata // 125))
    nd = 9 * 9 * 3 * 125
    one, el = 8 * 25 * nd, 8 * st.epmat.op_r.numel()
    monkeypatch.setattr(eph._GridOptKR, "PLANE_BYTES", 1 << 20, raising=False)
    free = el + 4 * quarter * one + 3
    monkeypatch.setattr(eph.core, "free_bytes", lambda _: free)
    seen = []
    plan = eph.core.plan_batch
    monkeypatch.setattr(eph.core, "plan_batch", lambda *a, **k: seen.append(a) or plan(*a, **k))
    loop = eph.OuterKLoop(st, nk_batch=None, nk_batch_cap=4)
    if planes == 0:
        assert loop.rr is None and loop.G is not None
        assert seen[0][2] == el
        return
    assert loop.rr.PLANES == planes
    held = 2 * planes * one
    assert loop.rr.plane_buffers() == 2 * planes and held <= quarter * one
    assert seen[0][0] == free and seen[0][2] == el + held
    assert eph._GridOptKR.PLANES == 8


def test_outer_k_planes_of_a_usual_size_ask_for_no_memory(monkeypatch):
    st = _setup(9, 3, (19, 2, 3))
    st.epmat.op_r = torch.zeros((125, 1))

    def never(_):
        raise AssertionError("free memory asked for")

    monkeypatch.setattr(eph.core, "free_bytes", never)
    assert eph.OuterKLoop(st, nk_batch=4).rr.PLANES == 8


def test_outer_q_reports_its_arithmetic_and_times_its_transforms(monkeypatch):
    """The staged loop keeps what the direct one has: the payload buffers, ft_timer and, as the outer-k loop, the
    arithmetic that the transforms run in beside the one asked for."""
    st = _setup(3, 3, (4, 2, 3))
    L = eph.L
    for staged, prec, used in ((True, L.PREC_FP32, L.PREC_FP32), (True, L.PREC_BF16X3, L.PREC_FP32),
                               (False, L.PREC_BF16X3, L.PREC_BF16X3)):
        loop = _outer_q(st, nq_tile=5, nk_batch=10, precision=prec, staged=staged, keep_ep=True)
        assert loop.precision_requested == loop.precision == prec
        assert loop.stage_precision == {"RR->Rq": used, "Rq->kq": used}
        assert loop.precision_overridden == (prec != used)
        assert loop.g2.shape[-3:] == (3, 2, 2) and loop.ep.shape == loop.g2.shape and loop.ep.is_complex()
        assert (loop.gk is None) == staged

    class Event:
        now = 0

        def __init__(self, enable_timing):
            assert enable_timing

        def record(self):
            Event.now += 1
            self.at = Event.now

    monkeypatch.setattr(torch.cuda, "Event", Event)
    loop = _outer_q(st, nq_tile=5, nk_batch=10)
    loop.ft_timer = []
    loop.run_qtile(0, 5)
    assert [n for _, _, n in loop.ft_timer] == [50, 50, 20]   # (k, q) of each of the three k batches: 24 k, 5 q
    assert all(a.at + 1 == b.at for a, b, _ in loop.ft_timer)


def test_unknown_precision_is_refused():
    """The staged kernels run in FP32 whatever is asked for, but what is asked for has to exist, as for the direct ones."""
    for nw in (5, 8):
        st = _setup(nw, 3, (4, 2, 3))
        st.epmat.op_r = torch.zeros((1, 1))
        for make in (lambda p: eph.OuterQLoop(st, nq_tile=2, precision=p), lambda p: eph.OuterKLoop(st, precision=p)):
            make(eph.L.PREC_BF16X3)
            with pytest.raises(eph.L.EphipError, match="precision"):
                make(7)
