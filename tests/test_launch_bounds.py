"""Entries whose launch would pass the 2^32 threads of a grid dimension refuse it (a launch past it may leave work out
without an error); argument checks only, no GPU."""
import ctypes as C

import pytest

from ephip import _lib as L


def test_bte_tables():
    with pytest.raises(L.EphipError, match="too many entries"):
        L.call("ephip_bte_tables", 1, 1, None, 1 << 26, None, 64, None, None, 5, None, None, None)
    with pytest.raises(L.EphipError, match="null device pointer"):   # just within
        L.call("ephip_bte_tables", 1, 1, None, (1 << 26) - 8, None, 64, None, None, 5, None, None, None)


def test_staged_rq_rotate():
    g = (C.c_int32 * 3)(256, 256, 256)
    for nk, msg in ((1 << 24, "too many"), ((1 << 24) - 1, "null device pointer")):   # times 16 q, 16 modes
        with pytest.raises(L.EphipError, match=msg):
            L.call("ephip_staged_rq_rotate", 4, 16, 2, 16, 0, nk, None, None, None, C.addressof(g), None, None, 4 * 16 * 16,
                   None, None, None, None, 1 << 24, None, None, None, None)
