"""mpic_last_timing: the FP32 form's deposit is its J gather, not what else a
step does beside it."""
import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd.workloads import courant_tau

pytestmark = pytest.mark.gpu


def test_deposit_is_the_gather_alone():
    """One marker in a flat box of 147456 tiles: push and gather are both
    launches with one tile to do, a few microseconds; the sort's scan reads
    every tile's counts (38 MB) and the E caps take a quarter of the nodes."""
    n, h = (768, 16, 768), (0.1,) * 3
    M = np.zeros(1, dtype=ma.MARKER_DTYPE)
    M["x"] = M["z"] = 38.4
    M["y"], M["rho"], M["qDivM"], M["id"] = 0.8, -1.0, -1.0, 1
    r = ma.Run(n, h, tuple(a * b for a, b in zip(n, h)), courant_tau(h), [ma.BC_OPEN] * 6, 0.0,
               precision=ma.FP32_SPLIT, max_markers=1)
    z = np.zeros(3 * r.nodes)
    r.set_fields(z, z)
    r.load_markers(M)
    r.init()
    r.advance(5)
    r.sync()
    for steps in (1, 2, 20):
        times = []
        for _ in range(5):
            r.advance(steps)
            times.append(r.timing())
        push, deposit, rest = np.median(times, axis=0) / steps
        print("per step: push %.4f ms, deposit %.4f, rest %.4f" % (push, deposit, rest))
        assert push > 0 and deposit > 0
        assert deposit <= 2 * push
        if steps > 1:                     # (one step has no following push to measure it by)
            assert rest > 2 * deposit
    r.close()
