"""Packing of marker records through an order with entries that name no record:
they are not followed, their positions are reported, and the other records are
those the order names.  The packing is called directly (no call of the public
interface leaves such an order)."""
import ctypes

import numpy as np
import pytest

import mandor3_amd as ma

pytestmark = pytest.mark.gpu
I, L, D, F, P = ctypes.c_int, ctypes.c_long, ctypes.c_double, ctypes.c_float, ctypes.c_void_p


def struct(*fields):
    return type("S", (ctypes.Structure,), {"_fields_": list(fields)})


# mpic_internal.h, mpic_readout.h
Grid = struct(("n", I * 3), ("GY", I), ("GZ", I), ("ncell", L), ("h", D * 3), ("tau", D))
NodeBlock = struct(("g", Grid), ("lo", I), ("d", I * 3), ("nc", I))
MarkerBlock = struct(("perm", P), ("extent", P), ("bad", P), ("words", I), ("nt", I * 3), ("h", D * 3),
                     ("qm", F * 8))
Readout = struct(("kind", I), ("words", L), ("dst", P), ("block", NodeBlock), ("mean", I), ("F", P * 3),
                 ("markers", MarkerBlock), ("m32", P * 3), ("m64", P * 9))
MARKERS32, MARKERS64 = 4, 5


class Device:
    """Device copies of arrays, freed together."""

    def __init__(self):
        self.lib, self.held = ma.lib(), []

    def put(self, a):
        a = np.ascontiguousarray(a)
        p = P()
        assert self.lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(a.nbytes)) == 0
        self.held.append(p)
        assert self.lib.hipMemcpy(p, P(a.ctypes.data), ctypes.c_size_t(a.nbytes), I(1)) == 0
        return p.value

    def close(self):
        for p in self.held:
            self.lib.hipFree(p)


@pytest.mark.parametrize("form", [MARKERS32, MARKERS64])
@pytest.mark.parametrize("words", [8, 7])
@pytest.mark.parametrize("count", [70, 40000])           # one slot, several
def test_entries_that_name_no_record(count, words, form):
    lib = ma.lib()
    ref, unref, readout = (getattr(lib, n) for n in (
        "_Z11readout_refv", "_Z13readout_unrefv", "_Z7readoutPK7ReadoutiiP12ihipStream_t"))
    readout.argtypes = [P, I, I, P]
    rng = np.random.default_rng(count)
    extent = count + 5
    perm = rng.permutation(extent)[:count].astype(np.int32)
    where = np.array([3, count // 2, count - 1])
    for bad in (None, -1, extent, 2 ** 31 - 1, -2 ** 31):
        p = perm.copy()
        if bad is not None:
            p[where] = bad
        d = Device()
        q = Readout()
        q.kind, q.words = form, count * words
        out = np.full((count, words), 2 ** 64 - 1, dtype=np.uint64)
        q.dst = out.ctypes.data
        report = P()
        assert lib.hipHostMalloc(ctypes.byref(report), ctypes.c_size_t(8), ctypes.c_uint(0)) == 0
        at = ctypes.cast(report, ctypes.POINTER(L))
        at[0] = -1
        q.markers.perm, q.markers.extent = d.put(p), d.put(np.array([extent], np.int32))
        q.markers.bad, q.markers.words = report.value, words
        q.markers.nt[:], q.markers.h[:] = (2, 2, 2), (1.0, 1.0, 1.0)
        ids = np.arange(1, extent + 1, dtype=np.int32)
        if form == MARKERS64:
            cols = rng.normal(0, 1, (6, extent))
            w = rng.normal(0, 1, (2, extent)).astype(np.float32)
            q.m64[:] = [d.put(c) for c in cols] + [d.put(c) for c in w] + [d.put(ids)]
            u = cols[3]
        else:
            pos = np.zeros((extent, 4), np.float32)      # cell word 0: key 0, species 0
            mom = rng.normal(0, 1, (extent, 4)).astype(np.float32)
            q.m32[:] = [d.put(pos), d.put(mom), d.put(ids)]
            u = mom[:, 0].astype(float)
        ref()
        try:
            assert readout(ctypes.addressof(q), 1, 0, None) == 0
            got = at[0]
        finally:
            unref()
            d.close()
            lib.hipHostFree(report)
        good = np.ones(count, bool)
        if bad is not None:
            good[where] = False
            assert got in where
            assert (out[where] == 0).all()
        else:
            assert got == -1
        assert np.array_equal(out[good, 3].view(np.float64), u[perm[good]])
        if words == 8:
            assert np.array_equal(out[good, 7].astype(np.int64), ids[perm[good]])
