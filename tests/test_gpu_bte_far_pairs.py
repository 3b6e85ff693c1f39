"""Scattering sums where both deltas of a pair vanish: nothing is added, whatever its g2, as in the per-term form."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("smearing", [1, 2])
def test_pairs_without_a_delta_add_nothing(backend, smearing):
    import torch
    from ephip import _lib as L
    f64, i32, i64 = (dict(dtype=t, device="cuda") for t in (torch.float64, torch.int32, torch.int64))
    nq = cs = 6
    es = torch.tensor([0.0, 0.01, 500.0], **f64)                  # the last state is out of reach of any Gaussian
    ikq = torch.tensor([1, 2, 1, 2, 2, 1], **i32)
    g2 = torch.tensor([[1.0], [float("inf")], [2.0], [float("nan")], [3.0], [1.5]], device="cuda")
    om = torch.full((nq, 1), 0.02, **f64)
    col, off, one, zero = torch.arange(cs, **i32), torch.arange(3, **i64), torch.ones(3, **i64), torch.zeros(2, **i64)
    mu, T, eta = torch.tensor([0.0], **f64), torch.tensor([0.03], **f64), torch.tensor([0.02], **f64)
    count = torch.tensor([cs], **i32)
    tq, ts = torch.empty(2 * nq, **f64), torch.empty(3, **f64)
    got = []
    for tables in (False, True):
        out, sin, code = torch.zeros(3, **f64), torch.full((cs,), 9.0, **f64), torch.zeros(cs, **i32)
        head = [L.ptr(x) for x in (count, col, ikq, g2, zero, off, one, one)]
        tail = [4, smearing, 1e-5, 3, L.ptr(zero), L.ptr(out), L.ptr(sin), L.ptr(code), L.stream_handle()]
        if tables:
            L.call("ephip_bte_tables", nq, 1, L.ptr(om), 3, L.ptr(es), 1, L.ptr(mu), L.ptr(T), 4, L.ptr(tq), L.ptr(ts),
                   L.stream_handle())
            L.call("ephip_bte_accumulate_tables", 1, cs, 1, 1, nq, *head, L.ptr(es), L.ptr(tq), L.ptr(ts), 0.1, 1,
                   L.ptr(T), L.ptr(eta), *tail)
        else:
            L.call("ephip_bte_accumulate_units", 1, cs, 1, 1, *head, L.ptr(es), L.ptr(om), 0.1, 1, L.ptr(mu), L.ptr(T),
                   L.ptr(eta), *tail)
        got.append(torch.cat([out, sin]))
    near = torch.isfinite(got[0])
    assert bool(near[:1].item()) == (smearing == 1)               # a Lorentzian reaches everywhere
    assert torch.equal(near, torch.isfinite(got[1]))
    # a few operations apart: rounding of the deltas' arguments and of the factors
    assert bool(((got[0] - got[1]).abs() <= 1e-12 * got[0].abs())[near].all())
