"""Results are read whatever HIP call of the caller's thread has failed before:
its error is the caller's, not the read-out's."""
import ctypes

import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("n", [8, 33])                   # one pinned slot, several
def test_results_after_a_failed_call(n, prec):
    st = workloads.two_stream_box(n)
    r = ma.Run(st["n"], st["h"], st["L"], st["tau"], st["bc"], 0.0, precision=prec,
               max_markers=st["markers"].size)
    z = np.zeros(3 * r.nodes)
    r.set_fields(z, z)
    r.load_markers(st["markers"])
    r.init()
    r.step(diag=False)
    reads = [r.fields, r.J, lambda: r.node_fields(0), r.markers, r.temperature]
    want = [f() for f in reads]
    for f, w in zip(reads, want):
        p = ctypes.c_void_p()
        assert ma.lib().hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 60)) != 0
        got = f()
        ma.lib().hipGetLastError()
        for x, y in zip(got, w):
            assert np.array_equal(x, y)
    r.close()
