"""The FP64 tiled push where its tiles end: partial tiles at the high faces, 4
and 8 wavefronts per tile, several batches per wavefront, and markers just
below the far face, whose cell rounds to n (their key is clamped into the box,
so they are pushed outside their tile's loop).  Positions and momenta bit for
bit against the oracle, fields to the J summation order."""
import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd.workloads import courant_tau
from oracle_lib import Oracle
from test_gpu_parity import by_id, rel_l2

pytestmark = pytest.mark.gpu
H = 0.05


def state(n, bc, ppc, edge, seed=3):
    rng = np.random.default_rng(seed)
    N = ppc * int(np.prod(n))
    M = np.zeros(N, dtype=ma.MARKER_DTYPE)
    for a, c in enumerate("xyz"):
        M[c] = rng.uniform(0, n[a] * H, N)
        M["v" + c] = rng.normal(0, 1.0, N)          # most markers cross a face, many two or three
    if edge:
        for a, c in enumerate("xyz"):
            M[c][a::7] = np.nextafter(n[a] * H, 0)
    M["rho"] = -1.0
    M["qDivM"] = -1.0
    M["id"] = np.arange(1, N + 1)
    nodes = 3 * int(np.prod([v + 1 for v in n]))
    return M, rng.normal(0, 0.3, nodes), rng.normal(0, 0.3, nodes)


@pytest.mark.parametrize("waves", ["4", "8"])
@pytest.mark.parametrize("n,ppc,bc", [((7, 8, 9), 40, 0), ((12, 13, 18), 6, 0), ((9, 10, 11), 30, 2),
                                      ((8, 11, 13), 12, 1)])
def test_tiles_at_the_faces(n, ppc, bc, waves, monkeypatch):
    monkeypatch.setenv("MPIC_TILE_WAVES", waves)
    edge = bc == 0
    M, E, F = state(n, bc, ppc, edge)
    if edge:
        # the reference's floor (int)(x/h + 128) - 128 takes them to cell n
        assert all((M[c][a::7] / H + 128.0 == n[a] + 128.0).all() for a, c in enumerate("xyz"))
    L = tuple(v * H for v in n)
    tau = courant_tau((H,) * 3)
    r = ma.Run(n, (H,) * 3, L, tau, (bc,) * 6, 0.0, max_markers=M.size)
    o = Oracle(n, (H,) * 3, L, tau, (bc,) * 6, 0.0)
    for s in (r, o):
        s.set_fields(E, F)
    r.load_markers(M)
    o.set_markers(M)
    r.init()
    o.init()
    r.step(diag=True)
    o.step()
    a, b = by_id(r.markers()), by_id(o.markers())
    assert np.array_equal(a["id"], b["id"])
    for f in ("x", "y", "z", "vx", "vy", "vz", "rho", "qDivM"):
        assert np.array_equal(a[f], b[f]), f
    # the sums of J in another order, its terms with fused multiply-adds
    for x, y in zip(r.fields(), o.fields()):
        assert rel_l2(x, y) < 1e-13
    r.close()
