"""Stages 2 and 3 of RR->kR with the k-side projection, one lane per (column, j), against 64-bit sums."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,rest,np_,lines,lda_pad", [
    (1, 1, 3, [[1]], 0), (3, 7, 5, [[1, 2], [], [3] * 5], 3), (4, 9, 7, [[1] * 9], 0), (5, 4, 3, [[4] * 3, [1]], 0),
    (8, 6, 7, [[2, 1, 1]] * 9, 1), (9, 3, 5, [[1]] * 6, 0), (12, 5, 5, [[1] * 4, [2] * 4, [1] * 5], 0),
    (13, 3, 7, [[3] * 50, [1] * 3], 0), (16, 2, 7, [[1] * 8] * 5, 5), (16, 3, 3, [[1]] * 300, 0)])
def test_lane_project(nw, rest, np_, lines, lda_pad):
    import torch
    from ephip import _lib as L
    rng = np.random.default_rng(nw + 10 * np_)
    h, dev = np_ // 2, "cuda"
    jl = 4 if nw <= 4 else 8 if nw <= 8 else 16
    nb = np.array([b for line in lines for b in line])              # bands of each k
    nk, nu, ng = len(nb), int(nb.sum()), nw * rest
    start = np.concatenate([[0], np.cumsum([len(x) for x in lines])]).astype(np.int32)
    line_of_k = np.repeat(np.arange(len(lines)), [len(x) for x in lines])
    x2 = rng.uniform(0, 1, len(lines))
    xk = np.stack([np.zeros(nk), x2[line_of_k], rng.uniform(0, 1, nk)], axis=1)
    kus = np.concatenate([[0], np.cumsum(nb)]).astype(np.int32)
    kpos = np.repeat(np.arange(nk), nb).astype(np.int32)
    band = np.concatenate([np.arange(b) for b in nb]).astype(np.int32) % nw
    U = (rng.standard_normal((nk, nw, nw)) + 1j * rng.standard_normal((nk, nw, nw))).astype(np.complex64)  # [k, band, j]
    split = len(lines) // 2                                          # two planes
    op1 = (rng.standard_normal((2, np_ * np_, ng * nw)) + 1j * rng.standard_normal((2, np_ * np_, ng * nw))).astype(
        np.complex64)

    def t(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev)

    d = dict(xk=t(xk), ls=t(start), kus=t(kus), kpos=t(kpos), state=t(kpos.astype(np.int64)), band=t(band), U=t(U),
             op=t(op1))
    us = torch.empty(len(lines) + 1, dtype=torch.int32, device=dev)
    c2 = torch.empty((len(lines), 8), device=dev)
    c3 = torch.full((nu + 4, 8), float("nan"), device=dev)
    uc = torch.full((nu + 4, jl), float("nan"), dtype=torch.complex64, device=dev)
    A = torch.zeros((nu, ng + lda_pad), dtype=torch.complex64, device=dev)
    s = L.stream_handle()
    L.call("ephip_lane_tables", nw, jl, np_, L.ptr(d["xk"]), 0, nk, 0, len(lines), L.ptr(d["ls"]), nu, L.ptr(d["kus"]),
           L.ptr(d["kpos"]), L.ptr(d["state"]), L.ptr(d["band"]), L.ptr(d["U"]), L.ptr(us), L.ptr(c2), L.ptr(c3),
           L.ptr(uc), s)
    ptrs = (C.c_void_p * 2)(*[d["op"][p].data_ptr() for p in range(2)])
    la, lz = (C.c_int32 * 2)(0, split), (C.c_int32 * 2)(split, len(lines))
    L.call("ephip_lane_project", nw, jl, ng, np_, 2, C.addressof(ptrs), C.addressof(la), C.addressof(lz), 0, L.ptr(us),
           L.ptr(c2), L.ptr(c3), L.ptr(uc), L.ptr(A), A.stride(0), s)
    got = A.cpu().numpy()
    assert (got[:, ng:] == 0).all()
    r = np.arange(-h, h + 1)
    op = op1.astype(np.complex128).reshape(2, np_, np_, rest, nw, nw)    # plane, c, b, rest, j, i
    for u in range(nu):
        k = kpos[u]
        e2, e3 = np.exp(2j * np.pi * xk[k, 1] * r), np.exp(2j * np.pi * xk[k, 2] * r)
        o = op[int(line_of_k[k] >= split)]
        w = U[k, band[u]].astype(np.complex128)
        ref = np.einsum("c,b,cbxji,j->xi", e3, e2, o, w).ravel()
        size = np.einsum("cbxji,j->xi", abs(o), abs(w)).ravel()
        # at most one rounding a step of the two folds (2 each), two sums of N, the product (2) and the sum over j,
        # in both parts; phases and their products rounded once each
        tol = 2 * (2 * np_ + 8 + nw) * 2.0 ** -24 * size
        assert (abs(got[u, :ng] - ref) <= tol).all(), (u, abs(got[u, :ng] - ref).max(), tol.min())


@pytest.mark.parametrize("box,staged,lanes", [(3, True, False), (5, True, True), (5, False, False)])
def test_lane_rule_keeps_the_digits_of_fp64_consumers(backend, box, staged, lanes):
    """27-R boxes and loops without the general staged kernels feed FP64 rates: same projection kernel as ever."""
    from ephip import _lib as L
    from ephip import eph
    from ephip import model as M
    m = M.make_model(nw=16, natoms=1, box_hd=3, box_g=box, seed=5, g_dtype=np.complex64)
    st = eph.setup_outer_q(m, (3, 3, 3), (3, 3, 3), (-0.3, 0.3), backend)
    assert 1 <= st.nbw <= 4
    loop = eph.OuterKLoop(st, nk_batch=8, staged=staged, precision=L.PREC_FP32)
    assert loop.rr.mfma and loop.rr.lanes() is lanes
