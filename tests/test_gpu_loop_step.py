"""The loop body's step (H over the whole step in one pass to the other H
buffer, caps and walls sharing launches with the sort) against the same step
through the stage calls, on every kind and mix of walls and on sizes where
rows and groups end differently.  Bit for bit where no J enters; with markers
positions and momenta of the first push bit for bit, fields to the J summation
order (FP32: the split form's bar of one step's rounding)."""
import itertools

import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd.workloads import courant_tau
from test_gpu_parity import by_id, rel_l2

pytestmark = pytest.mark.gpu
H = (0.05, 0.04, 0.06)
STAGES = ("em_h_half", "push_deposit", "em_h_step", "em_e_start", "j_finish", "em_e_finish")
WALLS = ["pp", "mm", "oo", "om", "mo"]
CODE = {"p": ma.BC_PERIODIC, "m": ma.BC_MIRROR, "o": ma.BC_OPEN}


def make(n, walls, prec, markers, seed, x=(0.0, 1.0)):
    rng = np.random.default_rng(seed)
    bc = [CODE[w[0]] for w in walls] + [CODE[w[1]] for w in walls]
    N = 3 * int(np.prod(n)) if markers else 0
    M = np.zeros(N, dtype=ma.MARKER_DTYPE)
    for a, c in enumerate("xyz"):
        M[c] = rng.uniform(0, n[a] * H[a], N)
        if a == 0:
            M[c] = x[0] * n[0] * H[0] + (x[1] - x[0]) * M[c]
        M["v" + c] = rng.normal(0, 0.5, N)
    M["rho"], M["qDivM"], M["id"] = -0.5, -1.0, np.arange(1, N + 1)
    nodes = 3 * int(np.prod([v + 1 for v in n]))
    E, F = rng.normal(0, 0.3, nodes), rng.normal(0, 0.3, nodes)
    out = []
    for _ in range(2):
        r = ma.Run(n, H, tuple(v * h for v, h in zip(n, H)), courant_tau(H), bc, 0.0, precision=prec,
                   max_markers=max(N, 1))
        r.set_fields(E, F)
        r.load_markers(M)
        r.init()
        out.append(r)
    return out


def staged(r):
    for s in STAGES:
        r.stage(s)


# every pair of wall kinds on neighbouring axes, on five sizes
MIXES = [(a, b, WALLS[(i + j) % 5]) for (i, a), (j, b) in itertools.product(enumerate(WALLS), repeat=2)]
SIZES = [(7, 7, 7), (8, 9, 10), (11, 7, 13), (9, 16, 8), (13, 10, 15)]


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("n", SIZES)
def test_vacuum_bit_exact_on_every_mix_of_walls(n, prec):
    for q, walls in enumerate(MIXES):
        a, b = make(n, walls, prec, False, q)
        for _ in range(3):
            a.step(diag=False)
            staged(b)
        # a stage step after loop steps, and the other way round
        staged(a)
        b.step(diag=False)
        for x, y in zip(a.fields(), b.fields()):
            assert np.isfinite(x).all() and np.array_equal(x, y), (n, walls)
        a.close()
        b.close()


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("walls", [("pp", "pp", "pp"), ("oo", "pp", "mm"), ("mo", "oo", "pp"), ("mm", "om", "oo")])
def test_with_markers(walls, prec):
    n = (13, 10, 15)
    a, b = make(n, walls, prec, True, 5)
    a.step(diag=False)
    b.stage(STAGES[0])
    we, wm = b.energy()
    b.stage(STAGES[1])
    wt = b.temperature()
    for s in STAGES[2:]:
        b.stage(s)
    # the same values summed in another order; FP32: a thread's partial in FP32
    np.testing.assert_allclose(a.diag_history(1)[0][1:], [we, wm, *wt],
                               rtol=1e-12 if prec == ma.FP64 else 1e-6)
    x, y = by_id(a.markers()), by_id(b.markers())
    assert np.array_equal(x["id"], y["id"])
    for f in ("x", "y", "z", "vx", "vy", "vz"):
        assert np.array_equal(x[f], y[f]), f
    for u, v in zip(a.fields(), b.fields()):
        assert rel_l2(u, v) < (1e-13 if prec == ma.FP64 else 1e-6)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
def test_graphs_after_sorts_and_stage_steps(prec):
    """Replays after calls that leave the double buffers at another phase."""
    n, walls = (13, 10, 15), ("oo", "pp", "mm")
    a, b = make(n, walls, prec, True, 9)
    a.set_graphs(True)
    for _ in range(2):
        a.advance(3)
        a.sort()
        a.advance(2)
        staged(a)
        a.advance(1)
    for _ in range(14):
        staged(b)
    x, y = by_id(a.markers()), by_id(b.markers())
    assert np.array_equal(x["id"], y["id"])
    for f in ("x", "y", "z"):
        np.testing.assert_allclose(x[f], y[f], rtol=0, atol=1e-12 if prec == ma.FP64 else 1e-5)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("n", [(32, 32, 16), (33, 32, 16), (36, 33, 29)])
def test_order_over_several_scan_workgroups(n, prec):
    """One scan workgroup of 256 tiles exactly, 288 and 648 tiles (two and
    three workgroups), a third of the tiles empty: every marker is in the order
    the loop's scan (FP32: in the gather's launch, in rounds of few registers)
    and rank leave exactly once, and the next push agrees with the stages'."""
    a, b = make(n, ("oo", "pp", "mm"), prec, True, 3, (0.3, 0.8))
    for _ in range(3):
        a.step(diag=False)
        staged(b)
    x, y = by_id(a.markers()), by_id(b.markers())
    assert np.array_equal(x["id"], np.unique(x["id"])) and np.array_equal(x["id"], y["id"])
    for f in ("x", "y", "z"):
        np.testing.assert_allclose(x[f], y[f], rtol=0, atol=1e-12 if prec == ma.FP64 else 1e-5)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
@pytest.mark.parametrize("walls", [("pp", "om", "mm"), ("mo", "pp", "oo")])
def test_vacuum_over_several_groups_of_edge_workgroups(walls, prec):
    """24 x 33 x 40: 27 workgroups of edge nodes, four groups of eight (the
    components' workgroups lie eight apart) with the last one partly empty."""
    a, b = make((24, 33, 40), walls, prec, False, 2)
    for _ in range(2):
        a.step(diag=False)
        staged(b)
    for x, y in zip(a.fields(), b.fields()):
        assert np.array_equal(x, y)
    a.close()
    b.close()
