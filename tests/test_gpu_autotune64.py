"""mpic_autotune on FP64 runs, whose shape it leaves alone: it reports it."""
import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd.workloads import courant_tau

pytestmark = pytest.mark.gpu


# 27 tiles: eight wavefronts, items of 512 markers; 1000 tiles: four, one item per tile
@pytest.mark.parametrize("n,want", [(12, (8, 512)), (40, (4, 0))])
def test_reports_the_shape_in_use(n, want):
    h = (0.1,) * 3
    r = ma.Run((n,) * 3, h, (n * 0.1,) * 3, courant_tau(h), (0,) * 6, 0.0, max_markers=1000)
    z = np.zeros(3 * r.nodes)
    r.set_fields(z, z)
    r.init()
    blocks, waves, item = r.autotune(steps=1)
    assert blocks > 0 and (waves, item) == want
    assert r.time == 0.0                  # nothing is timed
    r.close()


def test_untiled_run_has_neither(monkeypatch):
    monkeypatch.setenv("MPIC_UNTILED", "1")
    h = (0.1,) * 3
    r = ma.Run((12,) * 3, h, (1.2,) * 3, courant_tau(h), (0,) * 6, 0.0, max_markers=1000)
    z = np.zeros(3 * r.nodes)
    r.set_fields(z, z)
    r.init()
    assert r.autotune(steps=1)[1:] == (1, 0)
    r.close()
