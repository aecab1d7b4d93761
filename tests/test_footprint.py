"""mpic_footprint counts what a run allocates for its markers: two record
buffers, the keys, the order and the work items."""
import ctypes

import pytest

import mandor3_amd as ma


def footprint(n, cap, prec):
    c = ma.Config()
    c.n[:] = n
    c.h[:] = (0.1,) * 3
    c.L[:] = tuple(0.1 * v for v in n)
    c.tau, c.precision, c.max_markers = 0.05, prec, cap
    out = ctypes.c_size_t()
    assert ma.lib().mpic_footprint(ctypes.byref(c), ctypes.byref(out)) == 0
    return out.value


# FP64: 60-byte records; a box of at most 64 tiles has a 16-byte item per 512 markers
@pytest.mark.parametrize("n,prec,marker,item", [
    ((12, 12, 12), ma.FP64, 2 * 60 + 8, 16), ((16, 16, 16), ma.FP64, 2 * 60 + 8, 16),
    ((17, 16, 16), ma.FP64, 2 * 60 + 8, 0), ((12, 12, 12), ma.FP32_SPLIT, 2 * 36 + 8, 0)])
def test_marker_memory(n, prec, marker, item, monkeypatch):
    monkeypatch.delenv("MPIC_ITEM_MARKERS", raising=False)
    a, b = footprint(n, 51200, prec), footprint(n, 2 * 51200, prec)
    assert b - a == 51200 * marker + 100 * item
