"""FP32 push at a displacement of one cell in a step: tau / h rounds to 1 in
FP32 where one mesh step is far smaller than the other two, and a marker next
to its cell's face at the speed of light then ends on the face two cells on."""
import numpy as np
import pytest

import mandor3_amd as ma
from oracle_lib import Oracle
from test_gpu_parity import by_id, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_marker_moves_a_whole_cell(axis):
    n = (16, 17, 18)
    h = [1e4] * 3
    h[axis] = 1.0
    tau = 1.0 / np.sqrt(sum(1.0 / v ** 2 for v in h)) * (1 - 1e-12)
    assert np.float32(tau / h[axis]) == 1.0
    top = np.nextafter(np.float32(1), np.float32(0))       # the last offset of a cell
    c = "xyz"[axis]
    # offsets at and beside both faces, both directions, speeds up to c in FP32
    off = np.array([0.0, 2.0 ** -24, 2.0 ** -23, 0.25, 0.5, 1 - 2.0 ** -22, float(top)])
    u = np.array([3.0, 1e2, 1e4, 3e4, 1e5, 1e6, 3e7])
    off, u, sgn = (v.ravel() for v in np.meshgrid(off, u, [-1.0, 1.0], indexing="ij"))
    M = np.zeros(off.size, dtype=ma.MARKER_DTYPE)
    for a, d in enumerate("xyz"):
        # a few cells apart, inside the box and across its tiles
        M[d] = (5 + np.arange(off.size) % 6 + (off if a == axis else 0.5)) * h[a]
    M["v" + c] = sgn * u
    M["rho"], M["qDivM"], M["id"] = -1e-9, -1.0, np.arange(1, off.size + 1)
    L = tuple(a * b for a, b in zip(n, h))
    r = ma.Run(n, h, L, tau, (0,) * 6, 0.0, precision=ma.FP32_SPLIT, max_markers=M.size)
    o = Oracle(n, h, L, tau, (0,) * 6, 0.0)
    z = np.zeros(3 * r.nodes)
    for s in (r, o):
        s.set_fields(z, z)
    r.load_markers(M)
    o.set_markers(M)
    r.init()
    o.init()
    r.step(diag=False)
    o.step()
    a, b = by_id(r.markers()), by_id(o.markers())
    assert np.array_equal(a["id"], b["id"])
    # offset, displacement and their sum in FP32, each to 2^-24 of at most 2 cells
    assert np.abs(a[c] - b[c]).max() <= 4 * 2.0 ** -23 * h[axis]
    # E = -tau J: every marker's current to FP32's rounding of its terms
    E, F = r.fields()[0], o.fields()[0]
    assert np.linalg.norm(F) > 0 and rel_l2(E, F) <= 2e-5
    r.close()
