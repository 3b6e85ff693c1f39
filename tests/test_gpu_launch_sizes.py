"""Entries over many units at the largest unit count, where units times columns pass 2^32 threads: one unit has columns,
and its results are those of a call with it alone."""
import pytest

pytestmark = pytest.mark.gpu
NU = 65535


def _count(torch, nu, n):
    c = torch.zeros(nu, dtype=torch.int32, device="cuda")
    c[0] = n
    return c


@pytest.mark.parametrize("nw,nm,nbw,cs", [(2, 3, 2, 16 * 257), (32, 48, 4, 4 * 257)])   # columns of a workgroup: 16, 4
def test_rotate_kq_g2(backend, nw, nm, nbw, cs):
    import torch
    from ephip import _lib as L
    gen = torch.Generator(device="cuda").manual_seed(nw)
    G = torch.randn((cs, nw * nm), generator=gen, dtype=torch.complex64, device="cuda")
    U = torch.randn((3, nw, nw), generator=gen, dtype=torch.complex64, device="cuda")
    uph = torch.randn((5, nm, nm), generator=gen, dtype=torch.complex64, device="cuda")
    om = torch.rand((5, nm), generator=gen, dtype=torch.float64, device="cuda") + 0.5
    col = torch.arange(cs, dtype=torch.int32, device="cuda") % 5
    ikq = torch.arange(cs, dtype=torch.int32, device="cuda") % 3
    b0 = torch.ones(3, dtype=torch.int64, device="cuda")
    b1 = torch.tensor([nbw, 1, nbw], dtype=torch.int64, device="cuda")
    got = []
    for nu in (1, NU):
        g2 = torch.full((cs, nbw * nm), -1.0, device="cuda")
        count = _count(torch, nu, cs)
        L.call("ephip_eph_rotate_kq_g2", nw, nm, nbw, nu, cs, L.ptr(count), L.ptr(col), L.ptr(ikq), L.ptr(G), nw * nm,
               cs * nw * nm, L.ptr(U), L.ptr(b0), L.ptr(b1), L.ptr(uph), L.ptr(om), L.ptr(g2), None, L.stream_handle())
        got.append(g2)
    assert bool((got[0] >= 0).all()) and torch.equal(*got)


def test_bte_accumulate_tables(backend):
    import torch
    from ephip import _lib as L
    cs, nm, nst = 256 * 257, 2, 4
    gen = torch.Generator(device="cuda").manual_seed(1)
    kw = dict(dtype=torch.float64, device="cuda")
    i64 = dict(dtype=torch.int64, device="cuda")
    g2 = torch.rand((cs, nm), generator=gen, device="cuda")
    om, es = torch.rand((7, nm), generator=gen, **kw) * 0.05 + 0.01, torch.rand(nst, generator=gen, **kw)
    col = torch.arange(cs, dtype=torch.int32, device="cuda") % 7
    ikq = torch.arange(cs, dtype=torch.int32, device="cuda") % nst
    off, one = torch.arange(nst, **i64), torch.ones(nst, **i64)
    mu, T, eta = torch.tensor([0.4], **kw), torch.tensor([0.03], **kw), torch.tensor([0.1], **kw)
    tq, ts = torch.empty(2 * nm * 7, **kw), torch.empty(nst, **kw)
    L.call("ephip_bte_tables", 7, nm, L.ptr(om), nst, L.ptr(es), 1, L.ptr(mu), L.ptr(T), 5, L.ptr(tq), L.ptr(ts),
           L.stream_handle())
    got = []
    for nu in (1, NU):
        count, zero = _count(torch, nu, cs), torch.zeros(nu + 1, **i64)
        out, sin = torch.zeros(nst, **kw), torch.full((cs,), -1.0, **kw)
        code = torch.zeros(cs, dtype=torch.int32, device="cuda")
        L.call("ephip_bte_accumulate_tables", nu, cs, 1, nm, 7, L.ptr(count), L.ptr(col), L.ptr(ikq), L.ptr(g2),
               L.ptr(zero), L.ptr(off), L.ptr(one), L.ptr(one), L.ptr(es), L.ptr(tq), L.ptr(ts), 0.1, 1, L.ptr(T),
               L.ptr(eta), 5, 1, 0.0, nst, L.ptr(zero), L.ptr(out), L.ptr(sin), L.ptr(code), L.stream_handle())
        got.append((out, sin, code))
    assert bool((got[0][1] >= 0).all()) and torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][2], got[1][2])
    # positive terms added by atomics, in any order
    assert bool(((got[0][0] - got[1][0]).abs() <= cs * 1.2e-16 * got[0][0]).all()) and float(got[0][0][0]) > 0


def test_fourier_batched(backend):
    import torch
    from ephip import _lib as L
    n, nr, nd = 64 * 257, 5, 2
    gen = torch.Generator(device="cuda").manual_seed(2)
    op = torch.randn((nr, nd), generator=gen, dtype=torch.complex64, device="cuda")
    r = torch.randint(-2, 3, (nr, 3), generator=gen, dtype=torch.int32, device="cuda")
    xk = torch.rand((n, 3), generator=gen, dtype=torch.float64, device="cuda")
    got = []
    for nu in (1, NU):
        out = torch.zeros((n, nd), dtype=torch.complex64, device="cuda")
        count = _count(torch, nu, n)
        L.call("ephip_fourier_batched_c32", nd, nr, L.ptr(op), nd, 0, L.ptr(r), L.ptr(xk), nu, n, L.ptr(count), None, 0,
               L.ptr(out), nd, 0, L.PREC_FP32, L.stream_handle())
        got.append(out)
    assert float(got[0].abs().min()) > 0 and torch.equal(*got)


def test_fourier_c64_columns(backend):
    """More columns than a grid dimension has room for (6 threads each); the columns repeat 1021 points."""
    import numpy as np
    import torch
    from ephip import _lib as L
    n, m = 2 ** 32 // 6 + 100000, 1021
    op = torch.tensor([[0.6 - 0.8j]], dtype=torch.complex128, device="cuda")
    r = torch.tensor([[2, -1, 3]], dtype=torch.int32, device="cuda")
    x = np.random.default_rng(3).uniform(-1, 1, (m, 3))
    period = torch.from_numpy(x).to("cuda")
    xk = period.repeat(-(-n // m), 1)[:n].contiguous()
    out = torch.zeros(n, dtype=torch.complex128, device="cuda")
    L.call("ephip_fourier_c64", 1, 1, L.ptr(op), 1, L.ptr(r), n, L.ptr(xk), L.ptr(out), 1, L.stream_handle())
    ref = torch.from_numpy((0.6 - 0.8j) * np.exp(2j * np.pi * (x @ [2, -1, 3]))).to("cuda")
    whole = out[: n // m * m].view(-1, m)
    for row in (0, whole.shape[0] - 1):        # |t| < 6 cycles: 6 2 pi 2^-53 in the angle, a few ulp of the rest
        assert float((whole[row] - ref).abs().max()) <= 1e-14
    for a in range(0, whole.shape[0], 1 << 16):   # every repetition gives the same bits
        assert bool((torch.view_as_real(whole[a:a + (1 << 16)]) == torch.view_as_real(whole[0])).all())
    assert torch.equal(out[n // m * m:], whole[0][: n % m])
