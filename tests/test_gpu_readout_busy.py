"""Read-outs beside a busy run: a thread that reads a run with steps in flight
waits for that run alone, so a finished run is read and a new one created
meanwhile."""
import threading
import time

import numpy as np
import pytest

import mandor3_amd as ma
from mandor3_amd import workloads

pytestmark = pytest.mark.gpu


def box(n, prec, blocks=None, monkeypatch=None):
    """The two-stream box, its push on 'blocks' workgroups (one: a step of
    several milliseconds that leaves the rest of the GPU idle)."""
    if blocks:
        monkeypatch.setenv("MPIC_PUSH_BLOCKS", str(blocks))
    st = workloads.two_stream_box(n)
    r = ma.Run(st["n"], st["h"], st["L"], st["tau"], st["bc"], 0.0, precision=prec,
               max_markers=st["markers"].size)
    if blocks:
        monkeypatch.delenv("MPIC_PUSH_BLOCKS")
    rng = np.random.default_rng(n)
    E = rng.normal(0, 1e-3, 3 * r.nodes).astype(np.float32).astype(float)
    r.set_fields(E, 0 * E)
    r.load_markers(st["markers"])
    r.init()
    return r


# the busy run's and the finished one's results: in one slot, and in several
@pytest.mark.parametrize("n", [12, 32])
def test_finished_run_beside_a_busy_one(n, monkeypatch):
    busy = box(32, ma.FP32_SPLIT, 1, monkeypatch)
    done = box(n, ma.FP32_SPLIT)
    busy.node_fields(0)                   # (first uses: pinned slots, helper threads)
    want = done.fields()[0]
    assert np.abs(want).max() > 0
    busy.advance(2)
    busy.sync()
    t0 = time.time()
    busy.advance(5)
    busy.sync()
    step = (time.time() - t0) / 5
    busy.advance(1 + int(1.5 / max(step, 1e-3)))      # 1.5 s of steps, or 1500 steps
    reader = threading.Thread(target=busy.node_fields, args=(0,))
    reader.start()
    time.sleep(0.1)                       # the reader waits for the steps by now
    assert reader.is_alive()
    got = done.fields()[0]
    read_meanwhile = reader.is_alive()
    st = workloads.two_stream_box(8)
    new = ma.Run(st["n"], st["h"], st["L"], st["tau"], st["bc"], 0.0, precision=ma.FP32_SPLIT)
    made_meanwhile = reader.is_alive()
    reader.join()
    assert np.array_equal(got, want)
    assert read_meanwhile, "the read-out of a finished run waited for another run's steps"
    assert made_meanwhile, "mpic_create waited for another run's steps"
    for r in (busy, done, new):
        r.close()
