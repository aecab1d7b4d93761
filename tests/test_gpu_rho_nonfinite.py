"""Charge density with a marker whose charge is not finite: its own eight nodes
are not finite either, the rest are those of the other markers."""
import numpy as np
import pytest

import mandor3_amd as ma

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_other_cells_keep_their_charge(bad, prec):
    n, h = (9, 10, 11), (0.1, 0.2, 0.05)
    rng = np.random.default_rng(4)
    cells = np.array([(3, 3, c) for c in (2, 4, 6, 8)])     # in one wavefront, no node shared
    k = np.repeat(np.arange(4), 5)
    M = np.zeros(k.size, dtype=ma.MARKER_DTYPE)
    for a, c in enumerate("xyz"):
        M[c] = (cells[k, a] + rng.uniform(0.1, 0.9, k.size)) * h[a]
    M["rho"] = rng.uniform(0.5, 1, k.size)
    M["qDivM"], M["id"] = -1.0, np.arange(1, k.size + 1)

    def rho(M):
        r = ma.Run(n, h, tuple(a * b for a, b in zip(n, h)), 0.01, [ma.BC_OPEN] * 6, 0.0,
                   precision=prec, max_markers=M.size)
        z = np.zeros(3 * r.nodes)
        r.set_fields(z, z)
        r.load_markers(M)
        r.init()
        # nodes [0, n]: the fold at the walls copies inner nodes to the ghosts
        v = r.rho().reshape([a + 5 for a in n])[2:-2, 2:-2, 2:-2]
        r.close()
        return v

    want = rho(M)
    for cell in range(4):
        B = M.copy()
        B["rho"][5 * cell + 2] = bad
        got = rho(B)
        own = np.zeros(want.shape, bool)
        i, j, l = cells[cell]
        own[i:i + 2, j:j + 2, l:l + 2] = True
        assert not np.isfinite(got[own]).any()
        # five markers a cell, summed in any order
        assert np.abs(got[~own] - want[~own]).max() <= 8 * 2.0 ** -53 * np.abs(want[~own]).max()
