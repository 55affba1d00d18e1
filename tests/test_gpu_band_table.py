"""The slot search's table: one that is too small is doubled until the search
fits, and finds the same slots.

A frozen plan on a grid of several levels below a shallow input is made with a
first table of 16 and of 1024 cells and of the size its bands ask for.  Slots
and generated slots are equal, as are the terms applied; the blocks agree to
1e-13 of the largest (a job's segments are added in no fixed order)."""
import ctypes
import os

import numpy as np
import pytest

import mrchem_amd as mw  # noqa: F401  (loads the library the program is linked to)

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cxx", "band_table.so")


def _run(cells):
    fn = ctypes.CDLL(LIB).band_table
    slots, gen = ctypes.c_longlong(), ctypes.c_longlong()
    terms, nodes = ctypes.c_ulonglong(), ctypes.c_int(1 << 14)
    blocks = np.zeros((nodes.value, 512))
    rc = fn(ctypes.c_longlong(cells), ctypes.byref(slots), ctypes.byref(gen), ctypes.byref(terms),
            blocks.ctypes.data_as(ctypes.c_void_p), ctypes.byref(nodes))
    assert rc == 0
    return slots.value, gen.value, terms.value, blocks[:nodes.value]


def test_a_table_that_is_too_small_grows():
    want = _run(0)
    print("%d nodes, %d slots, %d of them generated, %d terms" % (len(want[3]), want[0], want[1], want[2]))
    assert want[0] > 1024 and want[1] > 0  # more than the small tables hold
    for cells in (16, 1024):
        got = _run(cells)
        assert got[:3] == want[:3]
        assert np.max(np.abs(got[3] - want[3])) <= 1e-13 * np.max(np.abs(want[3]))
