"""The VSP convolution where J is zero on most x planes: a slab away from both
x walls, drifting across tile boundaries so that the planes move from step to
step, through the loop step and through the stage calls, against the oracle."""
import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd.workloads import courant_tau
from oracle_lib import Oracle
from test_gpu_parity import by_id, rel_l2

pytestmark = pytest.mark.gpu
STAGES = ("em_h_half", "push_deposit", "em_h_step", "em_e_start", "j_finish", "em_e_finish")
H = (0.05, 0.04, 0.06)


# J nodes, fields: FP64 sums in another order; FP32 the split form's field bar
@pytest.mark.parametrize("prec,bar", [(ma.FP64, 1e-12), (ma.FP32_SPLIT, 1e-5)])
@pytest.mark.parametrize("how", ["loop", "stages"])
@pytest.mark.parametrize("drift", [1, -1])
def test_slab_away_from_the_walls(drift, how, prec, bar):
    n = (48, 10, 11)
    rng = np.random.default_rng(6)
    N = 3000
    M = np.zeros(N, dtype=ma.MARKER_DTYPE)
    # tiles 5 and 6 of 12 along x (cells 20 to 27): the planes are 17 to 31 of [-2, 50]
    M["x"] = rng.uniform(21, 27, N) * H[0]
    for a, c in ((1, "y"), (2, "z")):
        M[c] = rng.uniform(0, n[a] * H[a], N)
        M["v" + c] = rng.normal(0, 0.3, N)
    M["vx"] = drift * rng.uniform(2, 4, N)       # a tile in ten to twelve steps
    M["rho"], M["qDivM"], M["id"] = -0.5, -1.0, np.arange(1, N + 1)
    L = tuple(a * b for a, b in zip(n, H))
    bc = (2, 0, 1, 2, 0, 1)
    tau = courant_tau(H)
    r = ma.Run(n, H, L, tau, bc, 0.0, precision=prec, max_markers=N)
    o = Oracle(n, H, L, tau, bc, 0.0)
    E, F = rng.normal(0, 1e-2, (2, 3 * r.nodes))
    for s in (r, o):
        s.set_fields(E, F)
        s.set_vsp(0.8)
    r.load_markers(M)
    o.set_markers(M)
    r.init()
    o.init()
    planes = set()
    for step in range(16):
        if how == "loop":
            r.step(diag=False)
        else:
            for s in STAGES:
                r.stage(s)
        o.step()
        x, y = r.J(), o.J()
        assert np.isfinite(x).all()
        assert rel_l2(x, y) <= bar, step
        # a plane without current has exactly none
        x, y = (np.abs(v).reshape(n[0] + 5, -1).max(1) for v in (x, y))
        assert np.array_equal(x > 0, y > 0), step
        on = np.flatnonzero(y > 0)
        planes.add((on[0], on[-1]))
        assert on[0] > 6 and on[-1] < n[0] - 3
        for u, v in zip(r.fields(), o.fields()):
            assert rel_l2(u, v) <= bar, step
    assert len(planes) > 3
    assert np.array_equal(by_id(r.markers())["id"], by_id(o.markers())["id"])
    r.close()
