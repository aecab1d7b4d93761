"""Two lasers in one run: their planes are added one after the other, by
launches of their own, in the loop step (FP64: not fused with the E update) as
through the stage calls and in the oracle."""
import numpy as np
import pytest

import mandor3_amd as ma
from oracle_lib import MARKER_DTYPE, Oracle, load_fixture
from test_gpu_parity import by_id, rel_l2

pytestmark = pytest.mark.gpu
STAGES = ("em_h_half", "push_deposit", "em_h_step", "em_e_start", "j_finish", "em_e_finish")


def make(cls, fx, markers, **kw):
    s = cls(fx["n"], fx["h"], fx["L"], fx["tau"][0], fx["bc"], 0.0, **kw)
    rng = np.random.default_rng(8)
    z = rng.standard_normal((2, 3 * s.nodes)) * (1e-2 if markers else 1.0)
    s.set_fields(z[0], z[1])
    M = fx["M0"] if markers else np.zeros(0, MARKER_DTYPE)
    (s.load_markers if cls is ma.Run else s.set_markers)(M)
    p = np.array(fx["laser_params"], dtype=float)
    q = p * np.array([0.7, 1, 1, 1.3, 1, 0, 1]) + np.array([0, 0, 0, 0, 0.4, 0, 0])   # backwards
    q[1] = q[2] = 0.0                     # at its peak from the first step on
    for v in (p, q):
        s.add_laser(v, fx["laser_map"])
    s.init()
    return s


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("prec", [ma.FP64, ma.FP32_SPLIT])
def test_vacuum(prec, graphs):
    fx = load_fixture("laser_mur")
    r, o = make(ma.Run, fx, False, precision=prec), make(Oracle, fx, False)
    s = make(ma.Run, fx, False, precision=prec)
    r.set_graphs(graphs)
    for _ in range(12):
        r.advance(1)
        o.step()
        for q in STAGES:
            s.stage(q)
    for x, y, w in zip(r.fields(), o.fields(), s.fields()):
        if prec == ma.FP64:
            assert np.array_equal(x, y) and np.array_equal(w, y)
        else:
            assert rel_l2(x, y) < 3e-6 and rel_l2(w, y) < 3e-6
    assert r.time == o.time
    r.close()
    s.close()


@pytest.mark.parametrize("prec,bar", [(ma.FP64, 1e-12), (ma.FP32_SPLIT, 1e-5)])
def test_with_markers(prec, bar):
    fx = load_fixture("laser_mur")
    r = make(ma.Run, fx, True, precision=prec, max_markers=fx["M0"].size)
    o = make(Oracle, fx, True)
    for _ in range(10):
        r.step(diag=True)
        o.step()
    for x, y in zip(r.fields(), o.fields()):
        assert rel_l2(x, y) <= bar
    if prec == ma.FP64:
        assert np.array_equal(by_id(r.markers())["id"], by_id(o.markers())["id"])
    r.close()
