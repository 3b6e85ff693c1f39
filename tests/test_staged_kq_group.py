"""The workgroup of the staged kR->kq kernel for any hints (host choice, no GPU)."""
import ctypes as C
import itertools

import pytest

from ephip import _lib as L


@pytest.mark.parametrize("np_", [3, 4, 5, 6, 7, 8])
def test_group_holds_a_kept_q_with_every_band(np_):
    """The kernel takes a kept q while its entries and its line fit the group, so one with all nbw bands has to fit an
    empty one: its loop over the slab would not advance otherwise. Two entries a thread need a place for the line."""
    g = (C.c_int32 * 5)()
    for nw, nm, (m2, m3) in itertools.product((1, 3, 8, 9, 16, 17, 31, 32), (1, 3, 18, 47, 48), ((1, 1), (5, 64), (64, 64))):
        for nbw in sorted({1, min(2, nw), max(1, nw // 2), max(1, nw - 1), nw}):
            for cols, width in itertools.product((0.0, 1.0, 40.0, 4096.0, 1e30), (0.0, 1.0, 1.39, 1.6, 2.5, 32.0)):
                L.call("ephip_staged_kq_group", nw, nm, nbw, np_, m2, m3, cols, width, C.addressof(g))
                nq, nb, tb, nug, ls = g
                assert nq * tb >= -(-nbw // nb) + (nq > 1) and ls >= 1, (nw, nm, nbw, m2, m3, cols, width, list(g))
                assert nug >= 1 and tb * nug <= 512
